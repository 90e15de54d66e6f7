"""The fused out-projection + FFN of a 256-channel block (k_block_tail) at the edges of its 16-row blocks, of its widths
(inner 256 / 512 / 1280 and ff 256 / 1024 / 2048 in steps of 256) and of its blocks per 16 rows (1, 2, 4), beside widths that take the separate launches (ff 320,
inner 192), through a one-level flow estimator against the oracle. Tolerance: a chain of about 20 products and norms whose
longest f32 sum has 2048 terms, sqrt(2048) 2^-24 = 2.7e-6 each, roots of squares added: 1.3e-5; the GELU's fit adds 1.2e-7."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT, rel_err
from models import CosyModel, F16

pytestmark = pytest.mark.gpu
TOL = 1.3e-5


SMALL = (1, 7, 8, 9, 17)  # 2 T rows: a part of a block, one short of it, whole, one over, a third


@pytest.mark.parametrize("heads,ff,n_x,frames", [(8, 1024, 2, SMALL), (4, 256, 1, SMALL), (20, 512, 2, SMALL), (8, 2048, 1, SMALL),
                                                 (3, 1024, 1, SMALL), (8, 320, 2, SMALL)])
def test_block_tail_widths(hip, oracle, heads, ff, n_x, frames):
    m = CosyModel(60 + heads, M=8, C=256, heads=heads, head_dim=64, n_mid=1, n_x=n_x, ff=ff, wtype=F16)
    est = m.create(hip)
    rng = np.random.default_rng(ff)
    for T in frames:
        in0, x, tb = m.inputs(rng, T)
        hip.cosy_begin(est, T, in0)
        for _ in range(2):  # the captured step and its replay
            got = hip.cosy_step(est, x, tb, T, m.M)
            want = oracle.cosy_step(m.ox, T, m.with_x(in0, x), tb)
            assert rel_err(got, want) < TOL, (heads, ff, T, rel_err(got, want))
            x = rng.standard_normal(x.shape).astype(np.float32)
        hip.cosy_end(est)


@pytest.mark.parametrize("T", [512, 513, 1024, 1025])  # 64 tiles of 16 rows: 4 blocks each (all 256 of ws), 72 and 128: 2
def test_block_tail_lengths(hip, oracle, T):           # (all 128 counts), 136: 1
    m = CosyModel(64, M=8, C=256, heads=4, head_dim=64, n_mid=0, n_x=1, ff=1024, wtype=F16)
    est = m.create(hip)
    in0, x, tb = m.inputs(np.random.default_rng(T), T)
    hip.cosy_begin(est, T, in0)
    got = hip.cosy_step(est, x, tb, T, m.M)
    want = oracle.cosy_step(m.ox, T, m.with_x(in0, x), tb)
    assert rel_err(got, want) < TOL, (T, rel_err(got, want))
    for _ in range(3):  # replays: the counts are zero again, the parts added in their order
        assert np.array_equal(hip.cosy_step(est, x, tb, T, m.M), got)
    hip.cosy_end(est)


CHILD = r"""
import sys, numpy as np
sys.path[:0] = [ROOT, ROOT + "/oracle", ROOT + "/tests"]
from vox_amd import voxhip as hip
from models import CosyModel, F16
hip.init("hip:0")
m = CosyModel(64, M=8, C=256, heads=4, head_dim=64, n_mid=1, n_x=1, ff=1024, wtype=F16)
est = m.create(hip)
for T in (7, 512, 513, 1024, 1025):
    in0, x, tb = m.inputs(np.random.default_rng(T), T)
    hip.cosy_begin(est, T, in0)
    hip.cosy_step(est, x, tb, T, m.M)
    rows = [l.split() for l in hip.profile_report().splitlines()]
    print(T, *(f"{r[0].split('/')[1]}={r[1]}" for r in rows if r and "k_block_tail<" in r[0]), flush=True)
"""


def test_block_tail_parts():
    # which form each length of the test above takes, from the profile's launch counts (three blocks a step)
    r = subprocess.run([sys.executable, "-c", CHILD.replace("ROOT", repr(ROOT))], env=dict(os.environ, VOX_PROFILE="gpu"),
                       capture_output=True, text=True, timeout=180)
    assert r.returncode == 0, r.stderr[-3000:]
    lines = [l.split() for l in r.stdout.splitlines() if l[:1].isdigit()]
    seen, parts = {}, {}
    for T, *counts in lines:
        now = {c.split("=")[0]: int(c.split("=")[1]) for c in counts}
        parts[int(T)] = [(k, n - seen.get(k, 0)) for k, n in now.items() if n != seen.get(k, 0)]
        seen = now
    assert parts == {T: [(f"k_block_tail<{ns}>", 3)] for T, ns in ((7, 4), (512, 4), (513, 2), (1024, 2), (1025, 1))}, parts
