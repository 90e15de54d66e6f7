"""The reduce of a product's K slices (k_gemm_splitk_reduce) with four columns a thread and, where n is not a multiple of 4,
with one, through matmul, on few rows (one block, a partial one) and on many."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F16, BF16 = 1, 2


@pytest.mark.parametrize("wt", [F16, BF16])
@pytest.mark.parametrize("m,n,K", [(5, 1, 512), (9, 3, 3072), (64, 514, 1024), (9, 1026, 3072), (400, 1001, 512),  # one column
                                   (5, 4, 512), (33, 1024, 3072)])                                              # four
def test_splitk_reduce_columns(hip, wt, m, n, K):
    rng = np.random.default_rng(m + n + K)
    w16 = (rng.standard_normal((n, K)) * 0.05).astype(np.float16)
    if wt == F16:
        data, w = w16.view(np.uint16), w16.astype(np.float64)
    else:
        data = (w16.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        w = (data.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    b = rng.standard_normal(n).astype(np.float32)
    x = rng.standard_normal((m, K)).astype(np.float32)
    mat = hip.upload(hip.HostMat(wt, data, n, K, None, b))
    try:
        y = hip.matmul(mat, x)
    finally:
        hip.mat_free(mat)
    want = x.astype(np.float64) @ w.T + b
    # x keeps 2^-22 of its value as two halves (f32 products: 2^-24); at most K f32 roundings in a slice whose sum has K /
    # slices terms, 32 slice sums and the bias round once each
    bound = (np.abs(x).astype(np.float64) @ np.abs(w).T) * (2.0 ** -22 + (K / 8 + 40) * 2.0 ** -24) + 2.0 ** -23 * np.abs(want)
    err = np.abs(y - want)
    assert np.all(err <= bound), float(np.max(err / bound))
