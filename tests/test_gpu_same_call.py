"""A call gives the same bits whatever calls came before it: weight copies that one entry point lays out (F32 weights for
k_gemm_x3p, F16 weights for k_gemm_hh) are not what decides another's kernels."""
import numpy as np
import pytest

from models import F32, make_mat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,K", [(32, 512, 2048), (5, 96, 256), (200, 1026, 512)])
def test_matmul_dev_noalloc_before_and_after_matmul(hip, m, n, K):
    rng = np.random.default_rng(m)
    data, _, bias = make_mat(rng, F32, n, K, bias=True)
    x = rng.standard_normal((m, K)).astype(np.float32)
    h = hip.upload(hip.HostMat(F32, data, n, K, None, bias))
    dx, dy = hip.DevBuf(m * K * 4), hip.DevBuf(m * n * 4)
    dx.upload(x)

    def call():
        hip.matmul_dev_noalloc(h, dx, m, dy)
        hip.sync()
        return dy.download((m, n), np.float32)
    first = call()
    hip.matmul(h, x)  # lays the weights out
    assert np.array_equal(call(), first)
    dx.free()
    dy.free()
    hip.mat_free(h)
