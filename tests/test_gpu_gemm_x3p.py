"""The F32-weight GEMM on packed split-f16 weights (k_gemm_x3p) through matmul, at the edges of its tiles and plans:
64 x 64 tiles on full grids, 32 x 64 and 32 x 32 below, K slices and their reduce, ragged rows, columns and
K (whose padding holds zeros)."""
import numpy as np
import pytest

import models
import pyoracle as po
from conftest import rel_err

pytestmark = pytest.mark.gpu


def bound(x, w):
    """Per element: both operands keep 2^-22 of their value and the lo.lo product is dropped (3 x 2^-22 of sum |x w|), and
    each of the K / 32 steps and up to 32 slice sums rounds once in f32."""
    s = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    return s * (3 * 2.0 ** -22 + (w.shape[1] / 32 + 40) * 2.0 ** -24)


@pytest.mark.parametrize("m,n,K", [
    (5, 16, 8), (5, 1, 72), (33, 97, 40), (64, 64, 64),  # 32 x 32 tiles: one, ragged in n and K, exact
    (31, 130, 520), (65, 130, 1096), (8, 768, 5376),      # K slices: a last slice shorter than the others
    (257, 770, 136), (512, 448, 72),                      # 32 x 64 tiles
    (512, 1602, 96), (511, 1666, 200),                    # 64 x 64 tiles, ragged
])
def test_matmul_f32(hip, m, n, K):
    rng = np.random.default_rng(m * 7 + n + K)
    w = rng.standard_normal((n, K)).astype(np.float32) * 0.05
    b = rng.standard_normal(n).astype(np.float32)
    x = rng.standard_normal((m, K)).astype(np.float32)
    mat = hip.upload(hip.HostMat(0, w, n, K, None, b))
    try:
        y = hip.matmul(mat, x)
    finally:
        hip.mat_free(mat)
    want = x.astype(np.float64) @ w.astype(np.float64).T + b
    err = np.abs(y - want)
    assert np.all(err <= bound(x, w) + 2.0 ** -23 * np.abs(want)), float(np.max(err))


@pytest.mark.parametrize("m,n,K", [
    (33, 2753, 2048), (64, 4094, 2120), (33, 6081, 4096),  # 64 x 64 tiles in 5, 4 and 2 slices, a short last one
    (80, 2433, 2056), (400, 514, 5376),                    # 32 x 64 tiles, odd rows of them, in two slices
    (200, 1347, 3080),                                     # in three
    (64, 2113, 1096), (80, 2433, 2040)])                   # 66 tiles: three slices; K one step short of two
def test_matmul_f32_long_k(hip, m, n, K):
    test_matmul_f32(hip, m, n, K)


def test_codec_96_channels(hip, oracle):
    # a decoder whose last block has 96 channels at 6,656 rows a call: its convolutions fill the CUs with 64 x 64 tiles, the
    # first block of tiles of each reads the history
    cc = dict(models.CODEC_TINY, decoder_dim=384, upsample_rates=[8, 13])
    m = models.CodecModel(77, cc)
    codec = m.create(hip)
    rng = np.random.default_rng(5)
    st, ost = hip.codec_state_new(codec), po.CodecState(m.ox, 64)
    for F in (16, 16):
        z = (rng.standard_normal((F, cc["codebook_dim"])) * 0.5).astype(np.float32)
        got, want = hip.codec_forward(codec, st, z), po.codec_forward(ost, z)
        assert rel_err(got, want) < 1e-3, rel_err(got, want)
    hip.codec_state_free(st)


@pytest.mark.parametrize("cols", [68, 96, 100])
def test_conv_tiles_ragged_in_columns(hip, oracle, cols):
    # a DiT step whose grouped position convolutions fill the CUs (832 rows, 8 groups of `cols` channels) with 64 x 64 tiles whose
    # last columns are padding. Tolerance: 8 products in a chain, the longest sum 800 terms, roots of squares added, sqrt(8 x
    # 800) 2^-24 = 4.8e-6, three times that. An oracle that has lost the weights' lo halves in those convolutions is beyond it.
    tol = 1.5e-5

    def model(lossy):
        m = models.F5Model(50 + cols, 8 * cols, 1, 1, ff_mult=1, K=3, groups=8, wtype=models.F32)
        if lossy:
            m.ox = po.F5(m.dim, 1, 1, 64, 1, m.mel, m.text, m.pe, *(po.Mat(*m.mats[k]) for k in ("in_proj", "norm_out", "proj_out")),
                         [{k: po.Mat(*v) for k, v in b.items()} for b in m.blocks],
                         *(po.Conv((c[0] * 1024).astype(np.float16).astype(np.float32) / 1024, *c[1:]) for c in m.pos))
        return m
    m = model(False)
    h = m.create(hip)
    cat0, x, ts, rope = m.inputs(np.random.default_rng(cols), 1, 832)
    hip.f5_begin(h, 1, 832, cat0, rope)
    got = hip.f5_step(h, x, ts, 1, 832, m.mel)
    hip.f5_end(h)
    want = oracle.f5_step(m.ox, 1, 832, m.with_x(cat0, x, 1), ts, rope)
    lost = oracle.f5_step(model(True).ox, 1, 832, m.with_x(cat0, x, 1), ts, rope)
    assert rel_err(lost, want) > 2 * tol, rel_err(lost, want)
    assert rel_err(got, want) < tol, rel_err(got, want)


def test_overflow_flag(hip):
    # an activation beyond the f16 range fails the call; infinities and NaN pass through as the products give them
    w = np.eye(64, dtype=np.float32) * 0.5
    mat = hip.upload(hip.HostMat(0, w, 64, 64))
    x = np.ones((40, 64), np.float32)
    x[39, 63] = -65520.0
    with pytest.raises(hip.VoxHipError, match="f16 range"):
        hip.matmul(mat, x)
    x[39, 63] = 65504.0
    assert hip.matmul(mat, x)[39, 63] == 32752.0
    x[39, 63], x[3, 5] = np.inf, np.nan
    y = hip.matmul(mat, x)
    assert not np.isfinite(y[39]).any() and np.isnan(y[3]).all() and np.isfinite(np.delete(y, (3, 39), axis=0)).all()
    hip.mat_free(mat)
