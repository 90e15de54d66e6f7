"""The codec pre-transformer's attention (k_codec_attn) in its forms: head dims on both sides of 64, grouped heads, windows
shorter than a call (the ring wraps), longer than one pass of its values (24 keys per group) and than one of its scores (256
keys), through streams of calls against the oracle. Tolerance: the samples pass about 60 products and convolutions after it,
the longest f32 sum 256 terms, 256 ** 0.5 * 2^-24 = 9.5e-7 each: 6e-5; a key or value of a wrong slot is far above it."""
import numpy as np
import pytest

from models import CODEC_TINY, CodecModel
from test_gpu_codec import rel_err

pytestmark = pytest.mark.gpu
TOL = 6e-5


@pytest.mark.parametrize("hd,kvh,W", [(8, 2, 5), (64, 1, 3), (64, 4, 72), (96, 2, 72), (128, 4, 300)])
def test_codec_attention_windows(hip, oracle, hd, kvh, W):
    m = CodecModel(50 + hd, cc=dict(CODEC_TINY, head_dim=hd, num_attention_heads=4, num_key_value_heads=kvh, sliding_window=W))
    codec = m.create(hip)
    chunks = [16, 1, 15, 2] + [16] * (20 if W > 256 else 6) + [1, 3]
    z = oracle.codec_quantize(m.ox, m.codes(np.random.default_rng(hd), sum(chunks)))
    st, ost, f0 = hip.codec_state_new(codec), oracle.CodecState(m.ox), 0
    for n in chunks:
        got, want = hip.codec_forward(codec, st, z[f0:f0 + n]), oracle.codec_forward(ost, z[f0:f0 + n])
        assert rel_err(got, want) < TOL, (f0, n, rel_err(got, want))
        f0 += n
    hip.codec_state_free(st)
