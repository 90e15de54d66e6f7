"""A call gives the same bits whatever calls came before it: weight copies that one entry point lays out (F32 weights for
k_gemm_x3p, F16 weights for k_gemm_hh) are not what decides another's kernels."""
import numpy as np
import pytest

from models import F16, F32, Model, make_mat

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


def _build(hip, seed, wtype, head_type=F32):
    mdl = Model(seed, 2, 256, 4, 2, 64, 512, wtype=wtype, head_rows=96, head_type=head_type)
    return mdl, hip.xfmr_create(mdl.hx, "same"), hip.upload(mdl.head[1])


@pytest.mark.parametrize("wtype", [F16, F32])
@pytest.mark.parametrize("steps", [False, True])
def test_decode_before_and_after_a_prefill(hip, wtype, steps):
    # six rows of one sequence, or one row of each of six: f32-activation passes of 5 to 8 rows
    mdl, xf, head = _build(hip, 90 + wtype, wtype)
    rng = np.random.default_rng(1)
    x = rng.standard_normal((6, 256)).astype(np.float32)
    seqs = [hip.seq_create(xf, 32) for _ in range(6)]
    dx = hip.DevBuf(x.nbytes)
    dx.upload(x)
    rows = 6 if steps else 1

    def call():
        out, logits = hip.DevBuf(rows * 256 * 4), hip.DevBuf(rows * 96 * 4)  # buffers of its own: a graph of its own
        if steps:
            hip.decode_steps_dev(xf, seqs, [0] * 6, dx, out, head, logits)
        else:
            hip.decode_dev(xf, seqs[0], 0, dx, 6, out, head, logits)
        hip.sync()
        keep.append((out, logits))
        return out.download((rows, 256), np.float32), logits.download((rows, 96), np.float32)
    keep = []
    first = call()
    other = hip.seq_create(xf, 32)
    hip.forward(xf, other, 0, rng.standard_normal((9, 256)).astype(np.float32), 256, head=head)
    hip.matmul(head, x)
    for a, b in zip(call(), first):
        assert np.array_equal(a, b)
    for bufs in keep:
        for b in bufs:
            b.free()
    dx.free()


def test_forward_heads_before_and_after_matmul(hip):
    # the input projection of a prefill and the head of six sessions' steps, both F32, before and after voxhip_matmul on them
    mdl, xf, head = _build(hip, 97, F16)
    rng = np.random.default_rng(2)
    w, _, b = make_mat(rng, F32, 256, 128, bias=True)
    proj = hip.upload(hip.HostMat(F32, w, 256, 128, None, b))
    seq = hip.seq_create(xf, 32)
    seqs = [hip.seq_create(xf, 32) for _ in range(6)]
    xp = rng.standard_normal((9, 128)).astype(np.float32)
    xs = rng.standard_normal((6, 256)).astype(np.float32)

    def call():
        return hip.forward(xf, seq, 0, xp, 256, in_proj=proj, head=head) + hip.forward_steps(xf, seqs, [0] * 6, xs, 256, head=head)
    first = call()
    hip.matmul(proj, xp)
    hip.matmul(head, xs)
    for a, b in zip(call(), first):
        assert np.array_equal(a, b)
