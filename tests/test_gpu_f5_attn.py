"""The DiT's attention (k_f5_attn) in each of its forms, chosen by the number of 32- and 64-row blocks, at the edges of its
key tiles (64), query blocks (32, 64, 128 rows) and of v's 4-key stores (N off the fours), against the oracle. Tolerance:
about 12 products and norms in one block, the longest f32 sum 1024 terms (inner), sqrt(1024) 2^-24 = 1.9e-6 each, plus the
dropped lo x lo terms (2^-22 per product): 12 * (1.9e-6 + 2.4e-7) = 2.6e-5."""
import numpy as np
import pytest

from conftest import rel_err
from models import F5Model, F16, F32

pytestmark = pytest.mark.gpu
TOL = 2.6e-5


@pytest.mark.parametrize("wtype,heads,B,N", [
    (F16, 2, 1, 1), (F16, 2, 2, 15), (F16, 2, 1, 32), (F16, 2, 2, 33), (F16, 2, 1, 64), (F16, 2, 1, 65), (F16, 2, 2, 129),
    (F16, 2, 1, 200), (F32, 2, 2, 33), (F32, 2, 1, 68),   # 32-row blocks; F32: the row path's own store of q, k and v
    (F16, 16, 2, 257), (F16, 16, 2, 300), (F16, 16, 2, 512),   # 64-row blocks
    (F16, 16, 2, 513), (F16, 16, 2, 580), (F16, 16, 2, 640)])  # 128-row blocks
def test_f5_attn_forms(hip, oracle, wtype, heads, B, N):
    m = F5Model(95, 128, 1, heads, mel=20, text=32, K=7, groups=4, wtype=wtype)
    f5 = m.create(hip)
    rng = np.random.default_rng(N)
    cat0, x, ts, rope = m.inputs(rng, B, N)
    hip.f5_begin(f5, B, N, cat0, rope)
    got = hip.f5_step(f5, x, ts, B, N, m.mel)
    hip.f5_end(f5)
    want = oracle.f5_step(m.ox, B, N, m.with_x(cat0, x, B), ts, rope)
    assert rel_err(got, want) < TOL, rel_err(got, want)
