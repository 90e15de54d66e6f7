"""The fragment-order split-f16 GEMM (k_gemm_hh) at the edges of its tiles, through voxhip_bench_gemm_hh, against float64
on the same operands (tests/test_gpu_gemm_tiles.py holds the mid-size shapes). Tolerance: the products are exact in f32, so
an output's error is that of the f32 accumulation, K / 32 roundings of partial sums plus the MFMA's own within 32 columns:
(K / 32 + 32) 2^-24 of the sum of the magnitudes, taken whole as the bound."""
import numpy as np
import pytest

from test_gpu_gemm_tiles import _operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("m,n,K", [
    (1, 1, 64), (1, 130, 128), (15, 33, 64), (16, 64, 192), (17, 63, 128), (31, 4, 320), (32, 32, 64),
    (33, 65, 192), (63, 127, 64), (64, 128, 128), (65, 129, 192), (129, 257, 64),  # one past each tile, n off the fours
    (33, 100, 2112), (70, 72, 4864), (33, 101, 2112),                             # split K, a short last slice, n off the fours
    (640, 2052, 64), (1290, 1030, 64)])                                           # the grids of the wide tiles
def test_gemm_hh_edges(hip, m, n, K, q8):
    a, w = _operands(hip, m, n, K, q8)
    want = a @ w.T
    bound = (K / 32 + 32) * 2.0 ** -24 * (np.abs(a) @ np.abs(w).T)
    for tile in range(-1, 5):  # -1: K split as in the models
        got = hip.bench_gemm_hh(m, n, K, q8=q8, tile=tile, warmup=0, iters=1, out=True)[1]
        worst = float(np.max(np.abs(got - want) / bound))
        assert worst <= 1.0, (m, n, K, q8, tile, worst)
        if tile == -1:
            sliced = got
        elif tile == 0 and K >= 2112:  # the sums of slices round differently: K was split
            assert not np.array_equal(got, sliced)
