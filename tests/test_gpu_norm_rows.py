"""The row norms of fixed widths (k_norm_rows) beside the general kernel (k_f5_modulate, dim 320), through the Vocos head
(f32 rows, affine) and the DiT step (planes, modulation), at row counts around a block's 4 and 8 rows, against the oracle.
Tolerance: the longest sums are 3 dim terms in f32, sqrt(3 * 1024) 2^-24 = 3.3e-6 each, over the eight products and norms
of one block; a statistic taken in f32 or a wrong row misses it by far. A mel far from zero makes the first norm's rows
far from zero too, where their squares would cancel."""
import numpy as np
import pytest

from conftest import rel_err
from models import F5Model, F16, F32

pytestmark = pytest.mark.gpu
TOL = 8 * 3.3e-6


@pytest.mark.parametrize("dim", [256, 320, 512, 768, 1024])
def test_norm_rows_f32(hip, oracle, dim):
    m = F5Model(90 + dim, 128, 1, 2, mel=20, text=32, K=7, groups=4, wtype=F32, vocos=dict(dim=dim, inter=3 * dim, layers=1, out=34))
    f5 = m.create(hip)
    rng = np.random.default_rng(dim)
    for T, shift in ((1, 0.0), (3, 0.0), (4, 30.0), (5, 0.0), (9, 30.0), (17, 0.0)):
        mel = (rng.standard_normal((T, 20)) + shift).astype(np.float32)
        got, want = hip.f5_vocos(f5, mel), oracle.vocos_head(m.vox, mel)
        assert rel_err(got, want) < TOL, (dim, T, rel_err(got, want))


@pytest.mark.parametrize("dim", [256, 320, 512, 768, 1024])
@pytest.mark.parametrize("B,N", [(1, 3), (2, 17)])
def test_norm_rows_planes(hip, oracle, dim, B, N):
    m = F5Model(91 + dim, dim, 1, dim // 64, mel=20, text=32, K=7, groups=4, wtype=F16)
    f5 = m.create(hip)
    rng = np.random.default_rng(dim + N)
    cat0, x, ts, rope = m.inputs(rng, B, N)
    hip.f5_begin(f5, B, N, cat0, rope)
    got = hip.f5_step(f5, x, ts, B, N, m.mel)
    hip.f5_end(f5)
    assert rel_err(got, oracle.f5_step(m.ox, B, N, m.with_x(cat0, x, B), ts, rope)) < TOL
