"""The F32-weight GEMM on packed split-f16 weights (k_gemm_x3p) through matmul, at the edges of its tiles and plans:
64 x 64 and 64 x 96 tiles on full grids, 32 x 64 and 32 x 32 below, K slices and their reduce, ragged rows, columns and
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
    # a decoder whose last block has 96 channels at 6,656 rows a call: its convolutions fill the CUs with 64 x 96 tiles, the
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
