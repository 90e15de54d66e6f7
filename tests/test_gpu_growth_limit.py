"""Buffers that grow with a call: a call refused for want of room leaves the library as it was for the calls that fit."""
import numpy as np
import pytest

from conftest import rel_err
from models import F16, F5Model, Model

pytestmark = pytest.mark.gpu
TOL = 1e-3  # keys and values of 16 bits


def limit_to_use(hip, more):
    """The VRAM limit at what is in use without any weight copy (an allocation that fits in their place alone takes it), and so
    much more."""
    hip.lib().voxhip_set_vram_limit(int(hip.mem_info().used + 1))
    for bits in range(34, 10, -1):
        try:
            hip.DevBuf(1 << bits).free()
            break
        except hip.VoxHipError:
            pass
    hip.lib().voxhip_set_vram_limit(int(hip.mem_info().used + more))


def test_row_scratch_after_a_refused_growth(hip, oracle):
    mdl = Model(860, 2, 256, 4, 2, 64, 512, wtype=F16, head_rows=64)
    xf, head = hip.xfmr_create(mdl.hx, "t"), hip.upload(mdl.head[1])
    seq = hip.seq_create(xf, 1024)
    rng = np.random.default_rng(1)
    x = rng.standard_normal((600, 256)).astype(np.float32)
    hip.forward(xf, seq, 0, x[:16], 256, head=head)
    limit_to_use(hip, 1 << 20)
    try:
        with pytest.raises(hip.VoxHipError, match="VRAM limit"):
            hip.forward(xf, seq, 0, x, 256, head=head)  # 512 rows a pass: scratch of several MiB
        for rows in (1, 6, 16):
            kv = mdl.oracle_kv(1024)
            out, _ = hip.forward(xf, seq, 0, x[:rows], 256, head=head)
            assert rel_err(out, oracle.transformer_forward(mdl.ox, kv, x[:rows])) < TOL
        dx, dout = hip.DevBuf(256 * 4), hip.DevBuf(256 * 4)
        dx.upload(x[16:17])
        hip.decode_dev(xf, seq, 16, dx, 1, dout, head)
        hip.sync()
        want = oracle.transformer_forward(mdl.ox, kv, x[16:17])
        assert rel_err(dout.download((256,), np.float32), want) < TOL
        dx.free()
        dout.free()
    finally:
        hip.lib().voxhip_set_vram_limit(0)
    out, _ = hip.forward(xf, seq, 0, x, 256, head=head)
    assert rel_err(out, oracle.transformer_forward(mdl.ox, mdl.oracle_kv(1024), x)) < TOL


def test_vocoder_after_a_refused_length(hip, oracle):
    m = F5Model(861, 64, 1, 1, mel=20, wtype=F16, vocos=dict(dim=64, inter=128, layers=2, out=66))
    h = m.create(hip)
    mel = np.random.default_rng(2).standard_normal((20000, m.mel)).astype(np.float32)
    hip.f5_vocos(h, mel[:40])
    limit_to_use(hip, 1 << 20)
    try:
        with pytest.raises(hip.VoxHipError, match="VRAM limit"):
            hip.f5_vocos(h, mel)
        got = hip.f5_vocos(h, mel[:50])
    finally:
        hip.lib().voxhip_set_vram_limit(0)
    assert rel_err(got, oracle.vocos_head(m.vox, mel[:50])) < TOL
