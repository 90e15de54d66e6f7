"""What a speech engine has this backend do, as cases that can be timed and compared.

Each case is a pass through the public entry points of vox_amd.voxhip at the shapes of vox_amd.synth (synthetic
weights of the engine's models): the talker's and the LM's decode steps and prefills, the F5-TTS DiT step and its
vocoder, the CosyVoice2 flow estimator, the Qwen3-TTS codec decoder and the plain matrix product. `exact` restates
each path in 64-bit torch from the stored weights.

A program loads a model once and then feeds it inputs, so the models here are built once per process (`_model`) and a
state holds what belongs to one request: its inputs, its KV sequences, its begun step or its output buffers.
"""
import functools
import math
import weakref

import numpy as np
import torch

from vox_amd import synth
from vox_amd import voxhip as vh

DEV = "cuda:0"
DECODERS = {"talker_q8": synth.TALKER_0_6B, "talker_q4": synth.TALKER_1_7B_Q4, "lm_q8": synth.COSY_LM_0_5B}
WTYPES = {"f32": vh.F32, "f16": vh.F16, "bf16": vh.BF16, "q8": vh.Q8, "q4": vh.Q4}
# the matrices of the models above, as (rows, cols): talker q|k|v and gate, LM gate, DiT FFN, Vocos pointwise, text head
SHAPES = ((4096, 1024), (3072, 1024), (4864, 896), (2048, 1024), (1536, 512), (1026, 512), (6144, 2048), (1024, 3072))


def listed():
    return [
        # one token of the 0.6B talker, batch 1, 512 tokens into an utterance: the step an engine repeats 12.5 times a second
        {"name": "decode_talker_q8", "kind": "decode", "model": "talker_q8", "batch": 1, "kv": 512},
        # eight sessions of the 1.7B q4 talker in one step: a server under load
        {"name": "decode_talker_q4_x8", "kind": "decode", "model": "talker_q4", "batch": 8, "kv": 1024},
        # the LM's prompt (text and prompt speech tokens) before it generates
        {"name": "prefill_lm_512", "kind": "prefill", "model": "lm_q8", "rows": 512, "past": 0},
        # a short text prompt of the talker, a ragged number of rows
        {"name": "prefill_talker_61", "kind": "prefill", "model": "talker_q8", "rows": 61, "past": 0},
        # one flow-matching step of F5-TTS over 10.7 s of mel, both guidance passes
        {"name": "dit_2x1000", "kind": "dit", "batch": 2, "frames": 1000},
        # a short sentence without guidance
        {"name": "dit_1x333", "kind": "dit", "batch": 1, "frames": 333},
        # the vocoder's backbone and head over 10 s of mel
        {"name": "vocos_938", "kind": "vocos", "frames": 938},
        # one estimator step of the CosyVoice2 flow over an utterance of 256 speech tokens
        {"name": "flow_512", "kind": "flow", "frames": 512},
        # the same for a short streamed piece
        {"name": "flow_101", "kind": "flow", "frames": 101},
        # an utterance's codec frames decoded at once, 16 to a call
        {"name": "codec_48_by_16", "kind": "codec", "frames": 48, "chunk": 16},
        # two seconds of codec frames as a streaming talker produces them, one to a call
        {"name": "codec_25_by_1", "kind": "codec", "frames": 25, "chunk": 1},
        # the engine's own matmul hook on one row: the smallest call there is
        {"name": "matmul_q8_1", "kind": "matmul", "wtype": "q8", "rows": 3072, "cols": 1024, "m": 1},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(("decode", "prefill", "dit", "vocos", "flow", "codec", "matmul"))
    if kind == "decode":
        return {"kind": kind, "model": rng.choice(("talker_q8", "talker_q4", "lm_q8")), "batch": rng.choice((1, 1, 2, 3, 5, 7, 8)),
                "kv": size(3, 1500)}
    if kind == "prefill":
        return {"kind": kind, "model": rng.choice(("talker_q8", "lm_q8")), "rows": size(9, 600), "past": rng.choice((0, 0, size(1, 300)))}
    if kind == "dit":
        return {"kind": kind, "batch": rng.choice((1, 2)), "frames": size(65, 1000)}
    if kind == "vocos":
        return {"kind": kind, "frames": size(20, 1400)}
    if kind == "flow":
        return {"kind": kind, "frames": size(20, 700)}
    if kind == "codec":
        chunk = rng.choice((1, rng.randint(2, 16), 16))
        return {"kind": kind, "chunk": chunk, "frames": rng.randint(8, 24) if chunk == 1 else chunk * rng.randint(1, 3) + rng.randint(1, chunk)}
    rows, cols = rng.choice(SHAPES)
    return {"kind": "matmul", "wtype": rng.choice(tuple(WTYPES)), "rows": rows, "cols": cols, "m": size(1, 400)}


# ---------------------------------------------------------------- the models a program loads once
def _vec(rng, n, mean, sd):
    return (mean + sd * rng.standard_normal(n)).astype(np.float32)


class _Vocoder:
    """F5-TTS's DiT and Vocos with their host arrays kept; handle() gives an f5 handle of its own."""

    def __init__(self):
        c, v = synth.F5_DIT, synth.F5_VOCOS
        self.c, self.v = c, v
        rng = np.random.default_rng(0)
        D, ff, inner = c["dim"], c["dim"] * c["ff_mult"], c["heads"] * c["dim_head"]
        n = iter(range(0x5000, 0x7000))

        def mat(rows, cols):
            return vh.mat_synthetic(c["wtype"], rows, cols, 0, next(n), 0.0, 0.02, bias=True)
        self.in_proj, self.norm_out, self.proj_out = mat(D, 2 * c["mel"] + c["text"]), mat(2 * D, D), mat(c["mel"], D)
        self.blocks = [{"ada": mat(6 * D, D), "q": mat(inner, D), "k": mat(inner, D), "v": mat(inner, D), "o": mat(D, inner),
                        "ff1": mat(ff, D), "ff2": mat(D, ff)} for _ in range(c["depth"])]
        G, K = c["groups"], c["K"]
        self.pos = [((rng.standard_normal((G, D // G, K, D // G)) * 0.02).astype(np.float32), _vec(rng, D, 0, 0.02), D, D, K, G)
                    for _ in range(2)]
        VD, VI = v["dim"], v["inter"]
        self.voc = dict(dim=VD, inter=VI, out=v["out"],
                        embed=((rng.standard_normal((1, VD, 7, c["mel"])) * 0.02).astype(np.float32), _vec(rng, VD, 0, 0.02), c["mel"], VD, 7, 1),
                        ln_w=_vec(rng, VD, 1, 0.02), ln_b=_vec(rng, VD, 0, 0.02), fln_w=_vec(rng, VD, 1, 0.02), fln_b=_vec(rng, VD, 0, 0.02),
                        head=mat(v["out"], VD),
                        blocks=[dict(dw=((rng.standard_normal((VD, 7)) * 0.1).astype(np.float32), _vec(rng, VD, 0, 0.02), VD, VD, 7, VD),
                                     ln_w=_vec(rng, VD, 1, 0.02), ln_b=_vec(rng, VD, 0, 0.02), gamma=_vec(rng, VD, 0, 0.1),
                                     pw1=mat(VI, VD), pw2=mat(VD, VI)) for _ in range(v["layers"])])
        self.free = []

    def handle(self):
        if self.free:
            return self.free.pop()
        c = self.c
        return vh.f5_create(c["dim"], c["depth"], c["heads"], c["dim_head"], c["ff_mult"], c["mel"], c["text"], c["pe_attn_head"],
                            self.in_proj, self.norm_out, self.proj_out, self.blocks, self.pos[0], self.pos[1], vocos=self.voc)


class _Flow:
    """CosyVoice2's flow estimator with its host arrays kept; handle() gives an estimator handle of its own."""

    def __init__(self):
        c = self.c = synth.COSY_FLOW
        M, C, inner, FF = c["M"], c["C"], c["heads"] * c["head_dim"], c["ff"]
        rng = np.random.default_rng(0)
        n = iter(range(0x7000, 0x9000))

        def mat(rows, cols, bias):
            return vh.mat_synthetic(c["wtype"], rows, cols, 0, next(n), 0.0, 1.0 / math.sqrt(cols), bias=bias)

        def conv(cin, cout, K):
            return ((rng.standard_normal((cout, K, cin)) / math.sqrt(K * cin)).astype(np.float32), _vec(rng, cout, 0, 0.02), cin, cout, K, 1)

        def res(cin):
            return dict(c1=conv(cin, C, 3), c2=conv(C, C, 3), res=conv(cin, C, 1), n1w=_vec(rng, C, 1, 0.02), n1b=_vec(rng, C, 0, 0.02),
                        n2w=_vec(rng, C, 1, 0.02), n2b=_vec(rng, C, 0, 0.02))

        def xb():
            return dict(n1w=_vec(rng, C, 1, 0.02), n1b=_vec(rng, C, 0, 0.02), n3w=_vec(rng, C, 1, 0.02), n3b=_vec(rng, C, 0, 0.02),
                        q=mat(inner, C, False), k=mat(inner, C, False), v=mat(inner, C, False), o=mat(C, inner, True),
                        ff1=mat(FF, C, True), ff2=mat(C, FF, True), ff_dim=FF)
        self.down_res, self.up_res, self.mid_res = res(4 * M), res(2 * C), [res(C) for _ in range(c["n_mid"])]
        self.down_x, self.up_x = [xb() for _ in range(c["n_x"])], [xb() for _ in range(c["n_x"])]
        self.mid_x = [[xb() for _ in range(c["n_x"])] for _ in range(c["n_mid"])]
        self.down_conv, self.up_out, self.final_conv, self.final_proj = conv(C, C, 3), conv(C, C, 3), conv(C, C, 3), conv(C, M, 1)
        self.fn = (_vec(rng, C, 1, 0.02), _vec(rng, C, 0, 0.02))
        self.free = []

    def handle(self):
        if self.free:
            return self.free.pop()
        c = self.c
        return vh.cosy_create(c["M"], c["C"], c["heads"], c["head_dim"], self.down_res, self.up_res, self.mid_res, self.down_x, self.up_x,
                              self.mid_x, self.down_conv, self.up_out, self.final_conv, self.final_proj, *self.fn)


class _Codec:
    """Qwen3-TTS's codec decoder (f32 weights) with its host arrays and matrix handles kept."""

    def __init__(self):
        c = self.c = synth.QWEN3_CODEC
        rng = np.random.default_rng(0)
        n = iter(range(0x9000, 0xB000))
        CD, L, H, hd, I, dec = c["codebook_dim"], c["latent"], c["hidden"], c["head_dim"], c["inter"], c["dec"]
        qd, kd = c["heads"] * hd, c["kv_heads"] * hd

        def mat(rows, cols, std, bias):
            return vh.mat_synthetic(c["wtype"], rows, cols, 0, next(n), 0.0, std, bias=bias)

        def conv(K, cin, cout, dil=1, gain=1.0):
            return (mat(cout, K * cin, gain / math.sqrt(K * cin), True), K, cin, cout, dil)

        def snake(C):
            return (np.exp(_vec(rng, C, 0, 0.3)).astype(np.float32), (1.0 / (np.exp(_vec(rng, C, 0, 0.3)) + 1e-9)).astype(np.float32))
        self.pt_mats = [[mat(qd, H, H ** -0.5, False), mat(kd, H, H ** -0.5, False), mat(kd, H, H ** -0.5, False), mat(H, qd, qd ** -0.5, False),
                         mat(I, H, H ** -0.5, False), mat(I, H, H ** -0.5, False), mat(H, I, I ** -0.5, False)] for _ in range(c["layers"])]
        layers = [dict(ln1=_vec(rng, H, 1, 0.1), ln2=_vec(rng, H, 1, 0.1), attn_scale=_vec(rng, H, 0.01, 0.001),
                       mlp_scale=_vec(rng, H, 0.01, 0.001)) for _ in range(c["layers"])]
        inv = (1.0 / (10000.0 ** (np.arange(0, hd, 2, dtype=np.float64) / hd))).astype(np.float32)
        self.pt = dict(hidden=H, heads=c["heads"], kv_heads=c["kv_heads"], head_dim=hd, inter=I, eps=1e-5, theta=10000.0, window=c["window"],
                       inv_freq=inv, final_norm=_vec(rng, H, 1, 0.1), layers=layers)
        self.pre_conv, self.pt_in, self.pt_out = conv(3, CD, L), mat(H, L, L ** -0.5, True), mat(L, H, H ** -0.5, True)
        self.ups = [dict(tr=mat(r * L, L, L ** -0.5, False), K=r, tr_b=_vec(rng, L, 0, 0.02), dw_w=_vec(rng, L * 7, 0, 0.3), dw_b=_vec(rng, L, 0, 0.02),
                         dw_K=7, ln_w=_vec(rng, L, 1, 0.1), ln_b=_vec(rng, L, 0, 0.1), gamma=_vec(rng, L, 0, 0.1),
                         pw1=mat(4 * L, L, L ** -0.5, True), pw2=mat(L, 4 * L, (4 * L) ** -0.5, True)) for r in c["ratios"]]
        self.conv0 = conv(7, L, dec)
        self.blocks = []
        for b, r in enumerate(c["rates"]):
            i, o = dec >> b, dec >> (b + 1)
            self.blocks.append(dict(act=snake(i), tr=mat(2 * r * o, i, (2 * i) ** -0.5, False), K=2 * r, stride=r, cin=i, cout=o,
                                    tr_b=_vec(rng, o, 0, 0.02), a1=[snake(o) for _ in range(3)], a2=[snake(o) for _ in range(3)],
                                    c1=[conv(7, o, o, dil, 0.3) for dil in (1, 3, 9)], c2=[conv(1, o, o, 1, 0.3) for _ in range(3)]))
        last = dec >> len(c["rates"])
        self.final_act, self.final_conv = snake(last), conv(7, last, 1, 1, 0.1)
        self.codec = vh.codec_create(CD, L, self.pre_conv, self.pt_in, self.pt_out, self.pt, self.pt_mats, self.ups, self.conv0, self.blocks,
                                     self.final_act, self.final_conv)


@functools.lru_cache(maxsize=None)
def _model(name):
    vh.init("hip:0")
    if name in DECODERS:
        return synth.Decoder(dict(DECODERS[name], kv_len=0), capacity=64)
    return {"vocoder": _Vocoder, "flow": _Flow, "codec": _Codec}[name]()


@functools.lru_cache(maxsize=None)
def _matrix(wtype, rows, cols):
    vh.init("hip:0")
    return vh.mat_synthetic(WTYPES[wtype], rows, cols, 0, 0xB000 + rows + cols, 0.0, 0.02, bias=True)


class _State:
    """What one request holds; its sequences or its begun step go back when it is dropped."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


class _Buf:
    """A torch tensor as a device buffer of the binding."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def _release(kind, model, handle):
    if kind == "dit":
        vh.f5_end(handle)
    else:
        vh.cosy_end(handle)
    model.free.append(handle)


def _f5_rope(N, hd):
    inv = np.array([1.0 / 10000.0 ** (2 * j / hd) for j in range(hd // 2)], np.float32)
    a = (np.arange(N, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float32)
    return np.stack([np.cos(a), np.sin(a)], axis=-1).astype(np.float32)


def _inputs(case, seed):
    """The host arrays of one request, from the seed alone."""
    rng = np.random.default_rng(seed)

    def normal(*shape, sd=1.0):
        return (rng.standard_normal(shape) * sd).astype(np.float32)
    k = case["kind"]
    if k == "decode":
        return dict(x=normal(case["batch"], DECODERS[case["model"]]["hidden"]))
    if k == "prefill":
        return dict(x=normal(case["rows"], DECODERS[case["model"]]["hidden"]))
    if k == "dit":
        c = synth.F5_DIT
        B, N, mel = case["batch"], case["frames"], c["mel"]
        cat0 = normal(B * N, 2 * mel + c["text"])
        cat0[:, :mel] = 0.0
        return dict(cat0=cat0, x=normal(N, mel), ts=normal(c["dim"]), rope=_f5_rope(N, c["dim_head"]))
    if k == "vocos":
        return dict(mel=normal(case["frames"], synth.F5_DIT["mel"]))
    if k == "flow":
        c = synth.COSY_FLOW
        T, M = case["frames"], c["M"]
        in0 = np.zeros((2 * T, 4 * M), np.float32)
        in0[:T, M:] = normal(T, 3 * M)
        in0[:T, 2 * M:3 * M] = in0[0, 2 * M:3 * M]  # the speaker's vector, the same for every frame
        return dict(in0=in0, x=normal(T, M), tb=normal(2 + c["n_mid"], c["C"], sd=0.1))
    if k == "codec":
        return dict(z=normal(case["frames"], synth.QWEN3_CODEC["codebook_dim"], sd=0.5))
    return dict(x=normal(case["m"], case["cols"]))


def _sequences(case, seed, m, n, past, capacity):
    seqs = [vh.seq_create(m.xfmr, capacity) for _ in range(n)]
    for i, s in enumerate(seqs):
        if past:
            vh.seq_fill_synthetic(s, past, seed, 0xC0DE + i, 0.0, 1.0)
    return seqs


def prepare(case, seed):
    st = _State(case=case, **_inputs(case, seed))
    k = case["kind"]
    if k in ("decode", "prefill"):
        m = st.model = _model(case["model"])
        H = m.cfg["hidden"]
        if k == "decode":
            B, past = case["batch"], case["kv"]
            st.seqs = _sequences(case, seed, m, B, past, past + 64)
            st.pos = [past] * B
            st.d_x = _Buf(torch.from_numpy(st.x).to(DEV))
            st.d_out = _Buf(torch.zeros((B, H), device=DEV))
            st.d_logits = _Buf(torch.zeros((B, m.cfg["head_rows"]), device=DEV))
            st.d_token = _Buf(torch.zeros(B, dtype=torch.int32, device=DEV))
            st.cfgs = [vh.sample_cfg(0.9, 1.0, 50, seed=seed, frame=past, codebook=i) for i in range(B)]
            torch.cuda.synchronize()
        else:
            st.seqs = _sequences(case, seed, m, 1, case["past"], case["past"] + case["rows"] + 64)
        weakref.finalize(st, lambda seqs: [vh.seq_free(s) for s in seqs], st.seqs)
    elif k in ("dit", "flow"):
        m = st.model = _model("vocoder" if k == "dit" else "flow")
        st.handle = m.handle()
        if k == "dit":
            vh.f5_begin(st.handle, case["batch"], case["frames"], st.cat0, st.rope)
        else:
            vh.cosy_begin(st.handle, case["frames"], st.in0)
        weakref.finalize(st, _release, k, m, st.handle)
    elif k == "vocos":
        m = st.model = _model("vocoder")
        st.handle = m.handle()
        weakref.finalize(st, m.free.append, st.handle)
    elif k == "codec":
        st.model = _model("codec")
    else:
        st.mat = _matrix(case["wtype"], case["rows"], case["cols"])
    return st


def run(st):
    case = st.case
    k = case["kind"]
    if k == "decode":
        m = st.model
        if case["batch"] == 1:
            vh.decode_dev(m.xfmr, st.seqs[0], st.pos[0], st.d_x, 1, st.d_out, m.head, st.d_logits, st.cfgs[0], st.d_token)
        else:
            vh.decode_steps_dev(m.xfmr, st.seqs, st.pos, st.d_x, st.d_out, m.head, st.d_logits, st.cfgs, st.d_token)
        return {"hidden": st.d_out.t, "logits": st.d_logits.t, "token": st.d_token.t}
    if k == "prefill":
        m = st.model
        hidden, logits = vh.forward(m.xfmr, st.seqs[0], case["past"], st.x, m.cfg["hidden"], head=m.head)
        return {"hidden": hidden, "logits": logits}
    if k == "dit":
        return vh.f5_step(st.handle, st.x, st.ts, case["batch"], case["frames"], synth.F5_DIT["mel"])
    if k == "vocos":
        return vh.f5_vocos(st.handle, st.mel)
    if k == "flow":
        return vh.cosy_step(st.handle, st.x, st.tb, case["frames"], synth.COSY_FLOW["M"])
    if k == "codec":
        s = vh.codec_state_new(st.model.codec)
        pcm = [vh.codec_forward(st.model.codec, s, st.z[i:i + case["chunk"]]) for i in range(0, case["frames"], case["chunk"])]
        vh.codec_state_free(s)
        return np.concatenate(pcm)
    return vh.matmul(st.mat, st.x)


# ---------------------------------------------------------------- what a pass cannot do without
def _mat_bytes(t, rows, cols, bias=False):
    per = {vh.F32: 4.0, vh.F16: 2.0, vh.BF16: 2.0, vh.Q8: 1.0 + 4 / 32, vh.Q4: 0.5 + 4 / 32}[t]
    return rows * cols * per + (4 * rows if bias else 0)


def work(case):
    k = case["kind"]
    if k in ("decode", "prefill"):
        c = DECODERS[case["model"]]
        H, hd, I, L = c["hidden"], c["head_dim"], c["inter"], c["layers"]
        qd, kd = c["heads"] * hd, c["kv_heads"] * hd
        mats = ((qd + 2 * kd, H), (H, qd), (2 * I, H), (H, I))
        B, past, n = (case["batch"], case["kv"], 1) if k == "decode" else (1, case["past"], case["rows"])
        q4h = 2 / 32 if c.get("f16_scales") else 0  # f16 block scales are half of f32 ones
        body = sum(_mat_bytes(c["wtype"], r, cc) - q4h * r * cc for r, cc in mats)
        head = _mat_bytes(c["head_type"], c["head_rows"], H, c.get("head_bias", False))
        keys = sum(past + i + 1 for i in range(n))
        io = B * (n * H + H + c["head_rows"]) * 4
        return {"bytes": L * body + head + B * L * 2 * (past + n + n) * kd * 2 + io,
                "flops": B * (L * (n * 2 * sum(r * cc for r, cc in mats) + 4 * qd * keys) + 2 * c["head_rows"] * H)}
    if k == "dit":
        c = synth.F5_DIT
        D, inner, ff, mel, W = c["dim"], c["heads"] * c["dim_head"], c["dim"] * c["ff_mult"], c["mel"], 2 * c["mel"] + c["text"]
        B, N = case["batch"], case["frames"]
        R, lin = B * N, 4 * inner * D + 2 * ff * D
        weights = 2 * (c["depth"] * (lin + 6 * D * D) + 2 * D * D + W * D + mel * D) + 2 * 4 * D * c["K"] * (D // c["groups"])
        flops = c["depth"] * (2 * R * lin + 4 * B * N * N * inner + 12 * D * D) + 4 * R * D * c["K"] * (D // c["groups"]) + 2 * R * (W + mel) * D
        return {"bytes": weights + 4 * (R * W + N * mel + R * mel + N * c["dim_head"]), "flops": flops}
    if k == "vocos":
        v, mel, T = synth.F5_VOCOS, synth.F5_DIT["mel"], case["frames"]
        n = v["layers"] * 2 * v["dim"] * v["inter"] + v["out"] * v["dim"]
        e, d = v["dim"] * 7 * mel, v["layers"] * v["dim"] * 7
        return {"bytes": 2 * n + 4 * (e + d) + 4 * T * (mel + v["out"]), "flops": 2 * T * (n + e + d)}
    if k == "flow":
        c, T = synth.COSY_FLOW, case["frames"]
        M, C, inner, FF, R = c["M"], c["C"], c["heads"] * c["head_dim"], c["ff"], 2 * T
        res = sum(C * (3 * cin + 3 * C + cin) for cin in [4 * M, 2 * C] + [C] * c["n_mid"]) + 9 * C * C + M * C
        n_x = c["n_x"] * (2 + c["n_mid"])
        lin = n_x * (4 * inner * C + 2 * FF * C)
        return {"bytes": 4 * res + 2 * lin + 4 * (R * 4 * M + T * M + R * M), "flops": 2 * R * (res + lin) + n_x * 8 * T * T * inner}
    if k == "codec":
        c, F = synth.QWEN3_CODEC, case["frames"]
        CD, L, H, hd, I, dec = c["codebook_dim"], c["latent"], c["hidden"], c["head_dim"], c["inter"], c["dec"]
        qd, kd = c["heads"] * hd, c["kv_heads"] * hd
        per = [(3 * CD * L + 2 * L * H, 1), (c["layers"] * (H * (2 * qd + 2 * kd) + 3 * I * H), 1)]  # (weights, uses a frame)
        pos = 1
        for r in c["ratios"]:
            per.append((L * L * r, pos))
            pos *= r
            per.append((7 * L + 8 * L * L, pos))
        per.append((7 * L * dec, pos))
        ch = dec
        for r in c["rates"]:
            per.append((ch * (ch // 2) * 2 * r, pos))
            pos, ch = pos * r, ch // 2
            per.append((3 * 8 * ch * ch, pos))
        per.append((7 * ch, pos))
        calls = -(-F // case["chunk"])
        return {"bytes": calls * 4 * sum(w for w, _ in per) + 4 * F * (CD + pos),
                "flops": F * (2 * sum(w * p for w, p in per) + c["layers"] * 4 * min(F, c["window"]) * qd)}
    r, cc, m = case["rows"], case["cols"], case["m"]
    return {"bytes": _mat_bytes(WTYPES[case["wtype"]], r, cc, True) + 4 * m * (r + cc), "flops": 2 * m * r * cc}


def tolerance(case):
    k = case["kind"]
    if k == "decode":
        # each product's input is rounded to int8 per 32 values, so one last-place difference can move an input by 1/127
        # of its block and travels through the layers that follow (measured against 64 bits without that rounding: 0.014
        # for one session of the 28-layer q8 talker, 0.038 for q4)
        return {"rel": 0.02, "max": 0.3, "differ": 0.01}
    if k == "prefill":
        # the cache keeps keys and values in 16 bits: a last-place difference can move one by 2^-11 (hidden rows measured
        # 1.2e-4 off 64 bits over the talker's 28 layers, 6e-6 over the LM's 24); the talker's head takes the last row as int8
        return {"rel": 5e-3, "max": 0.1} if DECODERS[case["model"]]["head_type"] == vh.Q8 else {"rel": 1e-4, "max": 4e-3}
    return {"rel": 1e-5, "max": 4e-4}  # sums of 32 bits (measured 4e-7 to 1.6e-6 off 64 bits)


# ---------------------------------------------------------------- the same in 64 bits
def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV).double()


def _weights(mat, wtype):
    """A stored matrix as float64 (rows, cols) on the GPU, and its bias."""
    data, scale, bias = vh.mat_download(mat, wtype)
    d = torch.from_numpy(data.view(np.int16) if data.dtype == np.uint16 else data).to(DEV)
    if wtype == vh.F16:
        w = d.view(torch.float16).double()
    elif wtype == vh.BF16:
        w = d.view(torch.bfloat16).double()
    elif wtype == vh.F32:
        w = d.double()
    else:
        if wtype == vh.Q4:  # byte j of a block of 32: value j in the low half, value j + 16 in the high one, minus 8
            b = d.view(d.shape[0], -1, 16)
            d = torch.cat([b & 15, b >> 4], dim=2).reshape(d.shape[0], -1).double() - 8
        w = d.double().view(d.shape[0], -1, 32) * _t(scale)[:, :, None]
        w = w.reshape(d.shape[0], -1)
    return w, _t(bias)


def _lin(mat, wtype, x):
    w, b = _weights(mat, wtype)
    return x @ w.T + b


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _ln(x, w, b, eps):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + eps) * w + b


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))


def _mish(x):
    return x * torch.tanh(torch.nn.functional.softplus(x, threshold=40))


def _rotate_half(x, inv_freq, pos):
    """x (rows, heads, hd), pairs (i, i + hd / 2), at the f32 angles of the reference's table."""
    ang = (inv_freq[None, :] * pos.astype(np.float32)[:, None]).astype(np.float32)
    c, s = _t(np.cos(ang))[:, None], _t(np.sin(ang))[:, None]
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend(q, k, v, mask=None):
    """q (n, H, d) on keys k, v (t, KV, d) -> (n, H d)."""
    g = q.shape[1] // k.shape[1]
    out = []
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // g].T / math.sqrt(q.shape[2])
        if mask is not None:
            s = s.masked_fill(~mask, -math.inf)
        out.append(torch.softmax(s, -1) @ v[:, h // g])
    return torch.cat(out, dim=1)


def _exact_decoder(case, st):
    m, c = st.model, st.model.cfg
    hd, nh, nkv, eps = c["head_dim"], c["heads"], c["kv_heads"], c["eps"]
    many = case["kind"] == "decode"
    past, n = (case["kv"], case["batch"]) if many else (case["past"], case["rows"])
    pos = np.full(n, past) if many else past + np.arange(n)
    keys = [[vh.seq_download(s, li, past, nkv * hd) if past else None for s in st.seqs] for li in range(c["layers"])]
    mask = None if many else torch.arange(past + n, device=DEV)[None, :] <= torch.from_numpy(pos).to(DEV)[:, None]
    inv = m.inv_freq
    h = _t(st.x)
    for li in range(c["layers"]):
        ids, nm = m.mats[li], m.layers[li]
        y = _rms(h, _t(nm["ln1"]), eps)
        q, k, v = (_lin(ids[s], c["wtype"], y).view(n, -1, hd) for s in ("q", "k", "v"))
        if "qn" in nm:
            q, k = _rms(q, _t(nm["qn"]), eps), _rms(k, _t(nm["kn"]), eps)
        q, k = _rotate_half(q, inv, pos), _rotate_half(k, inv, pos).half().double()  # the cache keeps 16 bits
        v = v.half().double()
        cache = [None if kv is None else [_t(a).view(past, nkv, hd) for a in kv] for kv in keys[li]]

        def with_past(i, new):
            return [x if cache[i] is None else torch.cat([cache[i][j], x]) for j, x in enumerate(new)]
        if many:
            a = torch.cat([_attend(q[i:i + 1], *with_past(i, (k[i:i + 1], v[i:i + 1]))) for i in range(n)])
        else:
            a = _attend(q, *with_past(0, (k, v)), mask)
        h = h + _lin(ids["o"], c["wtype"], a)
        y = _rms(h, _t(nm["ln2"]), eps)
        h = h + _lin(ids["down"], c["wtype"], torch.nn.functional.silu(_lin(ids["gate"], c["wtype"], y)) * _lin(ids["up"], c["wtype"], y))
    out = _rms(h if many else h[-1:], _t(m.final_norm), eps)
    logits = _lin(m.head, c["head_type"], out)
    if many:
        return {"hidden": out, "logits": logits, "token": None}
    return {"hidden": out[0], "logits": logits[0]}


def _conv(x, w, b, left, right, dil=1):
    """x (T, cin) padded with zeros, w (cout, K, cin): y (T, cout)."""
    x = torch.nn.functional.pad(x, (0, 0, left, right))
    K = w.shape[1]
    T = x.shape[0] - (K - 1) * dil
    return sum(x[k * dil:k * dil + T] @ w[:, k].T for k in range(K)) + b


def _exact_dit(case, st):
    m, c = st.model, st.model.c
    D, H, hd, B, N, wt = c["dim"], c["heads"], c["dim_head"], case["batch"], case["frames"], c["wtype"]
    cat = st.cat0.copy()
    cat[:, :c["mel"]] = np.tile(st.x, (B, 1))
    ts = _t(st.ts)
    h = _lin(m.in_proj, wt, _t(cat))

    def pos_conv(x, cv):
        w, b = _t(cv[0]), _t(cv[1])
        g = D // c["groups"]
        return _mish(torch.cat([_conv(x[:, i * g:(i + 1) * g], w[i], 0, c["K"] // 2, c["K"] // 2) for i in range(c["groups"])], 1) + b)
    h = torch.cat([x + pos_conv(pos_conv(x, m.pos[0]), m.pos[1]) for x in h.view(B, N, D)])
    cos, sin = _t(st.rope[..., 0]).repeat(B, 1)[:, None], _t(st.rope[..., 1]).repeat(B, 1)[:, None]

    def turn(x):
        x = x.view(B * N, H, hd)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).view(B * N, H, hd)
    for blk in m.blocks:
        sh1, sc1, g1, sh2, sc2, g2 = _lin(blk["ada"], wt, ts[None])[0].view(6, D)
        y = _ln(h, 1 + sc1, sh1, 1e-6)
        q, k, v = turn(_lin(blk["q"], wt, y)), turn(_lin(blk["k"], wt, y)), _lin(blk["v"], wt, y).view(B * N, H, hd)
        a = torch.cat([_attend(q[i * N:(i + 1) * N], k[i * N:(i + 1) * N], v[i * N:(i + 1) * N]) for i in range(B)])
        h = h + g1 * _lin(blk["o"], wt, a)
        f = torch.nn.functional.gelu(_lin(blk["ff1"], wt, _ln(h, 1 + sc2, sh2, 1e-6)), approximate="tanh")
        h = h + g2 * _lin(blk["ff2"], wt, f)
    sc, sh = _lin(m.norm_out, wt, ts[None])[0].view(2, D)
    return _lin(m.proj_out, wt, _ln(h, 1 + sc, sh, 1e-6))


def _exact_vocos(case, st):
    v, wt = st.model.voc, st.model.c["wtype"]
    x = _conv(_t(st.mel), _t(v["embed"][0])[0], _t(v["embed"][1]), 3, 3)
    x = _ln(x, _t(v["ln_w"]), _t(v["ln_b"]), 1e-6)
    for b in v["blocks"]:
        p = torch.nn.functional.pad(x, (0, 0, 3, 3))
        w = _t(b["dw"][0])
        y = sum(p[k:k + x.shape[0]] * w[:, k] for k in range(7)) + _t(b["dw"][1])
        y = _gelu(_lin(b["pw1"], wt, _ln(y, _t(b["ln_w"]), _t(b["ln_b"]), 1e-6)))
        x = x + _t(b["gamma"]) * _lin(b["pw2"], wt, y)
    return _lin(v["head"], wt, _ln(x, _t(v["fln_w"]), _t(v["fln_b"]), 1e-6))


def _exact_flow(case, st):
    m, c, T = st.model, st.model.c, case["frames"]
    H, wt = c["heads"], c["wtype"]
    x = st.in0.copy()
    x[:, :c["M"]] = np.tile(st.x, (2, 1))
    x, tb = _t(x), _t(st.tb)

    def causal(cv, x):
        w, b = _t(cv[0]), _t(cv[1])
        return torch.cat([_conv(p, w, b, w.shape[1] - 1, 0) for p in (x[:T], x[T:])])

    def block(cv, w, b, x):
        return _mish(_ln(causal(cv, x), _t(w), _t(b), 1e-5))

    def resnet(r, x, t):
        return block(r["c2"], r["n2w"], r["n2b"], block(r["c1"], r["n1w"], r["n1b"], x) + t) + causal(r["res"], x)

    def xform(blocks, x):
        for p in blocks:
            y = _ln(x, _t(p["n1w"]), _t(p["n1b"]), 1e-5)
            q, k, v = (_lin(p[s], wt, y).view(2 * T, H, -1) for s in ("q", "k", "v"))
            x = x + _lin(p["o"], wt, torch.cat([_attend(q[i:i + T], k[i:i + T], v[i:i + T]) for i in (0, T)]))
            x = x + _lin(p["ff2"], wt, _gelu(_lin(p["ff1"], wt, _ln(x, _t(p["n3w"]), _t(p["n3b"]), 1e-5))))
        return x
    skip = xform(m.down_x, resnet(m.down_res, x, tb[0]))
    x = causal(m.down_conv, skip)
    for i, r in enumerate(m.mid_res):
        x = xform(m.mid_x[i], resnet(r, x, tb[1 + i]))
    x = xform(m.up_x, resnet(m.up_res, torch.cat([x, skip], 1), tb[1 + c["n_mid"]]))
    x = block(m.final_conv, *m.fn, causal(m.up_out, x))
    return causal(m.final_proj, x)


def _exact_codec(case, st):
    """The whole utterance at once: streaming it in any calls gives the same samples."""
    m, c, wt = st.model, st.model.c, st.model.c["wtype"]
    F, hd = case["frames"], c["head_dim"]

    def conv(cv, x):
        mat, K, cin, cout, dil = cv
        w, b = _weights(mat, wt)
        return _conv(x, w.view(cout, K, cin), b, (K - 1) * dil, 0, dil)

    def up(mat, bias, K, s, x):  # transposed convolution, causal: the last K - s rows belong to the next call
        y = (x @ _weights(mat, wt)[0].T).view(x.shape[0], K, -1)
        out = torch.zeros((x.shape[0] * s + K - s, y.shape[2]), dtype=torch.float64, device=DEV)
        for k in range(K):
            out[k:k + x.shape[0] * s:s] += y[:, k]
        return out[:x.shape[0] * s] + _t(bias)

    def snake(p, x):
        return x + _t(p[1]) * torch.sin(_t(p[0]) * x) ** 2
    h = _lin(m.pt_in, wt, conv(m.pre_conv, _t(st.z)))
    i = torch.arange(F, device=DEV)
    mask = (i[None, :] <= i[:, None]) & (i[None, :] > i[:, None] - c["window"])
    for ids, nm in zip(m.pt_mats, m.pt["layers"]):
        y = _rms(h, _t(nm["ln1"]), 1e-5)
        q, k, v = (_lin(ids[j], wt, y).view(F, -1, hd) for j in range(3))
        q, k = (_rotate_half(t, m.pt["inv_freq"], np.arange(F)) for t in (q, k))
        h = h + _t(nm["attn_scale"]) * _lin(ids[3], wt, _attend(q, k, v, mask))
        y = _rms(h, _t(nm["ln2"]), 1e-5)
        h = h + _t(nm["mlp_scale"]) * _lin(ids[6], wt, torch.nn.functional.silu(_lin(ids[4], wt, y)) * _lin(ids[5], wt, y))
    x = _lin(m.pt_out, wt, _rms(h, _t(m.pt["final_norm"]), 1e-5))
    for u in m.ups:
        y = up(u["tr"], u["tr_b"], u["K"], u["K"], x)
        w = _t(u["dw_w"]).view(-1, 7)
        p = torch.nn.functional.pad(y, (0, 0, 6, 0))
        d = sum(p[k:k + y.shape[0]] * w[:, k] for k in range(7)) + _t(u["dw_b"])
        x = y + _t(u["gamma"]) * _lin(u["pw2"], wt, _gelu(_lin(u["pw1"], wt, _ln(d, _t(u["ln_w"]), _t(u["ln_b"]), 1e-6))))
    x = conv(m.conv0, x)
    for b in m.blocks:
        x = up(b["tr"], b["tr_b"], b["K"], b["stride"], snake(b["act"], x))
        for j in range(3):
            x = x + conv(b["c2"][j], snake(b["a2"][j], conv(b["c1"][j], snake(b["a1"][j], x))))
    return conv(m.final_conv, snake(m.final_act, x))[:, 0].clamp(-1, 1)


def _exact_matmul(case, st):
    x = _t(st.x)
    if case["wtype"] == "q4" or case["wtype"] == "q8" and case["m"] <= 8:
        # these products take their inputs as int8 per 32 values: q = round(x / s), s = max / 127, both in 32 bits
        b = st.x.reshape(case["m"], -1, 32)
        s = np.abs(b).max(-1, keepdims=True) / np.float32(127)
        inv = np.where(s > 0, np.float32(1) / np.where(s > 0, s, np.float32(1)), np.float32(0)).astype(np.float32)
        x = (_t(np.rint(b * inv)) * _t(s)).reshape(case["m"], -1)
    return _lin(st.mat, WTYPES[case["wtype"]], x)


def exact(case, seed):
    st = prepare(case, seed)
    f = {"decode": _exact_decoder, "prefill": _exact_decoder, "dit": _exact_dit, "vocos": _exact_vocos, "flow": _exact_flow, "codec": _exact_codec,
         "matmul": _exact_matmul}[case["kind"]]
    return f(case, st)
