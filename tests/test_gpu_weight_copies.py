"""Weight copies (weights laid out again for the matrix cores) only take room that nothing else needs: a model that fits a
VRAM limit without them is created, begun and stepped under it, with the results it has elsewhere."""
import numpy as np
import pytest

from conftest import rel_err
import pyoracle as po
from models import F16, CodecModel, CosyModel, F5Model, Model

pytestmark = pytest.mark.gpu


def pack_f16(n, K):
    return (n + 15) // 16 * 16 * K * 2


def pack_x3(n, K):
    return (n + 15) // 16 * ((K + 31) // 32) * 2048


class Dit:
    """An F16 DiT: its step against the oracle, and the bytes of its copies (block linears; position convolutions)."""
    tol = 2e-5  # 12 products and norms in a chain, the longest sum 1024 terms: sqrt(12 x 1024) 2^-24 = 6.6e-6, three times that

    def __init__(self):
        self.m = F5Model(70, dim=512, depth=2, heads=8, ff_mult=2)
        self.linears = 2 * (pack_f16(1536, 512) + pack_f16(512, 512) + pack_f16(1024, 512) + pack_f16(512, 1024))
        self.others = 2 * 4 * pack_x3(128, 7 * 128)

    def create(self, hip):
        return self.m.create(hip)

    def begin(self, hip, h, oracle):
        self.args = self.m.inputs(np.random.default_rng(3), 2, 70)
        cat0, x, ts, rope = self.args
        hip.f5_begin(h, 2, 70, cat0, rope)
        self.want = oracle.f5_step(self.m.ox, 2, 70, self.m.with_x(cat0, x, 2), ts, rope)

    def step(self, hip, h):
        got = hip.f5_step(h, self.args[1], self.args[2], 2, 70, self.m.mel)
        assert rel_err(got, self.want) < self.tol, rel_err(got, self.want)
        return got

    def end(self, hip, h):
        hip.f5_end(h)


class Flow:
    """An F16 flow estimator of 256 channels (its blocks end in k_block_tail)."""
    tol = 2e-5  # 60 in a chain, the longest 1536 terms, of 0.1 of the rows each (residual adds): sqrt(60 x 1536) 2^-24 = 1.8e-5

    def __init__(self):
        self.m = CosyModel(71, M=8, C=256, heads=8, n_mid=2, n_x=2, ff=1024, wtype=F16)
        self.linears = 8 * (pack_f16(1536, 256) + pack_f16(256, 512) + pack_f16(1024, 256) + pack_f16(256, 1024))
        res = [sum(pack_x3(256, K) for K in (3 * cin, 768, cin)) for cin in (32, 512, 256, 256)]
        self.others = sum(res) + 3 * pack_x3(256, 768) + pack_x3(8, 256) + 256 * 16 * 256 * 4 + 128 * 4

    def create(self, hip):
        return self.m.create(hip)

    def begin(self, hip, h, oracle):
        self.args = self.m.inputs(np.random.default_rng(4), 90)
        in0, x, tb = self.args
        hip.cosy_begin(h, 90, in0)
        self.want = oracle.cosy_step(self.m.ox, 90, self.m.with_x(in0, x), tb)

    def step(self, hip, h):
        got = hip.cosy_step(h, self.args[1], self.args[2], 90, self.m.M)
        assert rel_err(got, self.want) < self.tol, rel_err(got, self.want)
        return got

    def end(self, hip, h):
        hip.cosy_end(h)


@pytest.fixture
def limit(hip):
    """Sets the VRAM limit to the bytes in use and so many more; none afterwards."""
    yield lambda more: hip.lib().voxhip_set_vram_limit(int(hip.mem_info().used + more))
    hip.lib().voxhip_set_vram_limit(0)


@pytest.mark.parametrize("kind", [Dit, Flow])
def test_create_gives_back_copies_that_do_not_all_fit(hip, oracle, limit, kind):
    c = kind()
    used = hip.mem_info().used
    c.create(hip)
    whole = hip.mem_info().used - used
    needed = whole - c.linears - c.others  # weights, stacked rows, vectors
    assert needed > 0
    limit(needed + 0.6 * c.linears)
    used = hip.mem_info().used
    h = c.create(hip)
    assert hip.mem_info().used - used == needed
    c.begin(hip, h, oracle)
    c.step(hip, h)
    c.end(hip, h)


@pytest.mark.parametrize("kind", [Dit, Flow])
def test_begin_takes_the_room_of_copies(hip, oracle, limit, kind):
    # a limit under which create finds room for every copy, and begin's buffers only in their place
    c = kind()
    used = hip.mem_info().used
    h = c.create(hip)
    whole = hip.mem_info().used - used
    c.begin(hip, h, oracle)
    c.step(hip, h)
    c.end(hip, h)
    limit(whole + (1 << 19))
    h = c.create(hip)
    full = hip.mem_info().used
    c.begin(hip, h, oracle)
    assert hip.mem_info().used < full - c.linears // 2
    first = c.step(hip, h)
    assert np.array_equal(c.step(hip, h), first)
    c.end(hip, h)
    hip.lib().voxhip_set_vram_limit(0)  # room again: the next begin lays the weights out again
    used = hip.mem_info().used
    c.begin(hip, h, oracle)
    assert hip.mem_info().used > used + c.linears
    c.step(hip, h)
    c.end(hip, h)


def test_allocation_takes_the_room_of_copies_in_use(hip, oracle, limit):
    # models with a begun step, captured graphs and states: an allocation that needs their copies' room gets it, and they go on
    dit, flow = Dit(), Flow()
    hd, hf = dit.create(hip), flow.create(hip)
    dit.begin(hip, hd, oracle)
    flow.begin(hip, hf, oracle)
    lm = Model(72, 2, 512, 8, 2, 64, 1024, wtype=F16, head_rows=96)
    xf, head = hip.xfmr_create(lm.hx, "copies"), hip.upload(lm.head[1])
    seq = hip.seq_create(xf, 64)
    x = np.random.default_rng(5).standard_normal((20, 512)).astype(np.float32)
    dec = CodecModel(73)
    codec = dec.create(hip)
    z = (np.random.default_rng(6).standard_normal((8, dec.cc["codebook_dim"])) * 0.5).astype(np.float32)
    pcm = po.codec_forward(po.CodecState(dec.ox, 64), z)

    def all_steps(st):
        dit.step(hip, hd)
        flow.step(hip, hf)
        out, logits = hip.forward(xf, seq, 0, x, 512, head=head)
        assert rel_err(out, oracle.transformer_forward(lm.ox, lm.oracle_kv(64), x)) < 1e-3
        got = np.concatenate([hip.codec_forward(codec, st, z[i:i + 2]) for i in (0, 2, 4, 6)])
        assert rel_err(got, pcm) < 1e-4, rel_err(got, pcm)
    st = [hip.codec_state_new(codec) for _ in range(2)]
    for _ in range(3):  # eager, captured, replayed
        dit.step(hip, hd)
        flow.step(hip, hf)
        hip.forward(xf, seq, 0, x, 512, head=head)
    all_steps(st[0])
    limit(1 << 19)
    used = hip.mem_info().used
    big = hip.DevBuf(dit.linears + flow.linears)  # fits in the copies' place alone
    assert hip.mem_info().used < used + (1 << 19)
    all_steps(st[1])
    with pytest.raises(hip.VoxHipError, match="VRAM limit"):
        hip.DevBuf(64 << 20)  # nothing left to give back
    big.free()
    dit.end(hip, hd)
    flow.end(hip, hf)
    for s in st:
        hip.codec_state_free(s)


def test_allocation_past_every_copy_leaves_them(hip, oracle, limit):
    dit = Dit()
    h = dit.create(hip)
    dit.begin(hip, h, oracle)
    first = dit.step(hip, h)
    limit(0)
    used = hip.mem_info().used
    with pytest.raises(hip.VoxHipError, match="VRAM limit"):
        hip.DevBuf(1 << 40)
    hip.lib().voxhip_set_vram_limit(0)
    with pytest.raises(hip.VoxHipError, match="hipMalloc"):
        hip.DevBuf(1 << 42)
    assert hip.mem_info().used == used
    assert np.array_equal(dit.step(hip, h), first)
    dit.end(hip, h)
