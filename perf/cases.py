"""The work that a user of this backend has it do, as cases that can be timed and compared.

A case is one pass through the C ABI (qp_dispatch, qp_graph_launch) in the op sequences that the JavaScript engine
issues (quipullm_amd/js/transformer.js): a one-token decode step replayed from a captured graph, a prompt chunk
dispatched op by op, the mixture-of-experts FFN of a prompt chunk, or the output head with the sampler's device part.
Bindings and uniforms are packed once, as the engine's bind groups are.  Models are a few layers deep: every layer of
a model runs the same ops, and the weights of two layers of the larger shapes with their output matrix already exceed
the last-level cache.

Weights are random GGUF blocks with zero mean and a standard deviation of about 1/sqrt(K), so that activations and
attention scores are of a real model's order; embeddings are N(0, 1); cached keys and values are N(0, 1).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from quipullm_amd import capi

F32, Q8, Q2, Q3, Q4, Q5, Q6, IQ4 = (capi.F32, capi.Q8_0, capi.Q2_K, capi.Q3_K, capi.Q4_K, capi.Q5_K, capi.Q6_K,
                                    capi.IQ4_NL)
NAME = capi.FMT_NAME
KQ = (Q2, Q3, Q4, Q5, Q6)
MIXED = (Q4, Q6)             # formats that share one GEMV launch
PLANAR = (Q8, IQ4)           # two bindings: quants, scales
STORE, ACC, SWIGLU, ARGMAX = capi.STORE, capi.ACC, capi.SWIGLU, capi.ARGMAX

# Weight types of a model file: the default and the tensors that differ (the usual mixes, and the plain ones).
MIX = {
    "q4km": (Q4, {"v": Q6, "down": Q6, "out": Q6}),
    "q5km": (Q5, {"v": Q6, "down": Q6, "out": Q6}),
    "q3k": (Q3, {"v": Q5, "out": Q6}),
    "q2k": (Q2, {"down": Q3, "out": Q6}),
    "q4k": (Q4, {}),
    "q6k": (Q6, {}),
    "q8": (Q8, {}),
    "iq4nl": (IQ4, {}),
    "f32": (F32, {"out": Q8}),
}


def fmt_of(case, tensor):
    default, other = MIX[case["mix"]]
    return other.get(tensor, default)


# ------------------------------------------------------------------------------------------------------- the cases
def _dense(kind, mix, D, nh, nkv, hd, F, **kw):
    return dict(kind=kind, mix=mix, D=D, nh=nh, nkv=nkv, hd=hd, F=F, **kw)


_8B = dict(D=4096, nh=32, nkv=8, hd=128, F=14336)
_TINY = dict(D=1024, nh=16, nkv=16, hd=64, F=2816)
_MOE = dict(D=2048, nh=32, nkv=4, hd=128, F=0, E=128, used=8, ffe=768)
_WIN = dict(D=2560, nh=16, nkv=8, hd=128, F=8192)


def listed():
    return [
        # a whole small chat model in Q8_0 answering token by token, f32 cache: launches and latency are all it costs
        _dense("decode", "q8", **_TINY, layers=8, vocab=32000, T=1, pos=96, ctx=512, f16=0, name="decode_tiny_q8"),
        # the 8B shape answering after a long prompt, f16 cache: the headline workload's layers and output matrix
        _dense("decode", "q4km", **_8B, layers=2, vocab=128256, T=1, pos=4100, ctx=4400, f16=1,
               name="decode_8b_q4km_ctx4k"),
        # the same step of a 128-expert mixture (8 used per token)
        _dense("decode", "q4k", **_MOE, layers=2, vocab=151936, T=1, pos=2051, ctx=2400, f16=1, qk=1,
               name="decode_moe_q4k_ctx2k"),
        # one token of a sliding-window model (one windowed and one global layer), which decodes op by op, f32 cache
        _dense("prefill", "q4km", **_WIN, layers=2, window=1024, T=1, pos=3001, ctx=4096, batch=32, f16=0, qk=1,
               name="decode_window_q4km_ctx3k"),
        # sampling from a large vocabulary: output matrix, penalties, top-k candidates
        _dense("sample", "q4km", **_8B, vocab=128256, topk=40, T=1, name="sample_head_128k"),
        # a prompt chunk in the engine's default setting (32 tokens per pass, f32 cache) inside a conversation
        _dense("prefill", "q4km", **_8B, layers=1, T=32, pos=480, ctx=4096, batch=32, f16=0,
               name="prefill_8b_q4km_32"),
        # a long prompt in one pass of 2048 tokens with the f16 cache: throughput
        _dense("prefill", "q4km", **_8B, layers=1, T=2048, pos=0, ctx=4400, batch=2048, f16=1,
               name="prefill_8b_q4km_2048"),
        # an ordinary prompt of odd length in another weight type, behind a cached prefix, f32 cache
        _dense("prefill", "q5km", **_8B, layers=1, T=333, pos=1000, ctx=4096, batch=512, f16=0,
               name="prefill_8b_q5km_333"),
        # a short question to the small Q8_0 model
        _dense("prefill", "q8", **_TINY, layers=2, T=77, pos=0, ctx=512, batch=128, f16=0, name="prefill_tiny_q8_77"),
        # a prompt chunk of the sliding-window model, its ring cache wrapping
        _dense("prefill", "q4km", **_WIN, layers=2, window=1024, T=500, pos=2100, ctx=4096, batch=512, f16=0, qk=1,
               name="prefill_window_q4km_500"),
        # the expert FFN of a long prompt, and of the default 32-token pass
        _dense("moe", "q4k", **_MOE, layers=1, T=2048, name="moe_ffn_q4k_2048"),
        _dense("moe", "q4k", **_MOE, layers=1, T=32, name="moe_ffn_q4k_32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "window", "moe", "sample"])
    hd = rng.choice([64, 128])
    nkv = rng.choice([2, 4, 8])
    group = rng.choice([1, 2, 4, 8])
    D = 256 * _log_int(rng, 2, 16)
    while nkv * group * hd > min(2 * D, 4096) or nkv * group * hd % 256:
        nkv, group = rng.choice([2, 4, 8]), rng.choice([1, 2, 4, 8])
    F = 256 * max(3, min(56, round(D / 256 * rng.uniform(2.0, 3.5))))
    shape = dict(D=D, nh=nkv * group, nkv=nkv, hd=hd, F=F)
    mix = rng.choice(["q4km", "q4km", "q5km", "q3k", "q2k", "q6k", "q8", "iq4nl", "f32"])
    f16 = rng.choice([0, 1])
    if kind == "decode":
        pos = _log_int(rng, 8, 8000)
        vocab = _log_int(rng, 8000, 130000)
        if rng.random() < 0.3:
            shape.update(F=0, E=rng.choice([16, 64, 128]), used=rng.choice([2, 4, 8]), ffe=256 * rng.randint(1, 4))
            mix = rng.choice(["q4k", "q6k"])
        return _dense("decode", mix, **shape, layers=rng.randint(1, 3), vocab=vocab, T=1, pos=pos,
                      ctx=pos + rng.randint(1, 600), f16=f16, qk=rng.choice([0, 1]))
    if kind == "sample":
        return _dense("sample", mix, **shape, vocab=_log_int(rng, 5000, 150000), topk=rng.choice([5, 20, 40, 64]), T=1)
    T = _log_int(rng, 2, 2048 if f16 and mix != "f32" else 700)
    if kind == "moe":
        shape.update(D=256 * rng.randint(4, 10), F=0, E=rng.choice([16, 64, 128]), used=rng.choice([2, 4, 8]),
                     ffe=256 * rng.randint(1, 3))
        return _dense("moe", rng.choice(["q4k", "q4k", "q5km", "q6k", "q8", "iq4nl"]), **shape, layers=1, T=T)
    pos = rng.choice([0, _log_int(rng, 10, 2000)])
    case = _dense("prefill", mix, **shape, layers=1, T=T, pos=pos, ctx=pos + T + rng.randint(0, 500),
                  batch=rng.choice([32, 512, 2048]), f16=f16, qk=rng.choice([0, 1]))
    case["batch"] = max(case["batch"], T)
    if kind == "window":
        case.update(layers=2, window=rng.choice([128, 512, 1024]), T=rng.choice([1, min(T, 700)]), qk=1)
    return case


# ------------------------------------------------------------------------------------------- weights, as GGUF blocks
_IQ4_TABLE = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
_BYTES = {F32: (1, 4), Q8: (32, 34), Q2: (256, 84), Q3: (256, 110), Q4: (256, 144), Q5: (256, 176), Q6: (256, 210),
          IQ4: (32, 18)}


def _halves(x):
    """f16 values as two columns of bytes."""
    return x.half().view(torch.uint8).reshape(-1, 2)


def gen_matrix(g, fmt, N, K):
    """Random blocks (uint8 [blocks, bytes]) of an N x K matrix with zero mean and deviation about 1/sqrt(K)."""
    std = 1.0 / math.sqrt(K)
    if fmt == F32:
        return torch.randn(N, K, generator=g, device="cuda").mul_(std).reshape(-1, 1).view(torch.uint8)
    per, size = _BYTES[fmt]
    nb = N * K // per
    raw = torch.randint(0, 256, (nb, size), generator=g, device="cuda", dtype=torch.uint8)
    spread = 0.75 + 0.5 * torch.rand(nb, generator=g, device="cuda")   # block scales differ by up to 5/3
    if fmt == Q8:
        raw[:, :2] = _halves(spread * std / 73.9)
    elif fmt == IQ4:
        raw[:, :2] = _halves(spread * std / 70.0)
    elif fmt == Q6:
        raw[:, 192:208] = (raw[:, 192:208].int() % 96 + 32).to(torch.uint8)   # scales 32 .. 127
        raw[:, 208:] = _halves(spread * std / (82.0 * 18.5))
    elif fmt == Q3:
        raw[:, 108:] = _halves(spread * std / (18.5 * 2.35))
    elif fmt == Q2:
        sc = raw[:, :16] & 15
        raw[:, :16] = sc | (sc << 4)
        d = (spread * std / (8.8 * 1.12)).half()
        raw[:, 80:82] = _halves(d)
        raw[:, 82:84] = _halves(d.float() * 1.5)
    else:
        mean, dev = (7.5, 4.6) if fmt == Q4 else (15.5, 9.2)
        d = (spread * std / (36.4 * dev)).half()
        raw[:, :2] = _halves(d)
        raw[:, 2:4] = _halves(d.float() * mean)
        sc = torch.randint(0, 64, (nb, 8), generator=g, device="cuda", dtype=torch.uint8)   # scales and mins alike
        lo, hi = sc[:, :4], sc[:, 4:]
        raw[:, 4:8] = raw[:, 8:12] = lo | ((hi >> 4) << 6)
        raw[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
    return raw


def dequant(raw, fmt, K):
    """The rows of the blocks `raw` in 64 bits, from the public GGUF block layouts."""
    if fmt == F32:
        return raw.reshape(-1).view(torch.float32).reshape(-1, K).double()

    def f16(a, b):
        return raw[:, a:b].contiguous().view(torch.float16).double().reshape(-1)

    n = raw.shape[0]
    r = raw.to(torch.int16)
    if fmt == Q8:
        return (raw[:, 2:].contiguous().view(torch.int8).double() * f16(0, 2)[:, None]).reshape(-1, K)
    if fmt == IQ4:
        t = torch.tensor(_IQ4_TABLE, dtype=torch.float64, device=raw.device)
        q = torch.cat([r[:, 2:] & 15, r[:, 2:] >> 4], 1).long()
        return (t[q] * f16(0, 2)[:, None]).reshape(-1, K)
    if fmt in (Q4, Q5):
        s = r[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = r[:, size_qs(fmt):].reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if fmt == Q5:
            bit = torch.arange(8, device=raw.device, dtype=torch.int16).reshape(1, 8, 1)
            q = q + 16 * ((r[:, 16:48].reshape(n, 1, 32) >> bit) & 1)
        w = (f16(0, 2)[:, None] * sc)[:, :, None] * q - (f16(2, 4)[:, None] * mn)[:, :, None]
        return w.reshape(-1, K)
    if fmt == Q6:
        ql, qh = r[:, :128].reshape(n, 2, 2, 32), r[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)                                       # [n, half, quarter, 32]
        shift = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.int16).reshape(1, 1, 4, 1)
        q = (lo | (((qh >> shift) & 3) << 4)) - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double() * f16(208, 210)[:, None]
        return (q.reshape(n, 16, 16).double() * sc[:, :, None]).reshape(-1, K)
    shift = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.int16).reshape(1, 1, 4, 1)
    if fmt == Q2:
        q = (r[:, 16:80].reshape(n, 2, 1, 32) >> shift) & 3
        sc = r[:, :16]
        w = (f16(80, 82)[:, None] * (sc & 15))[:, :, None] * q.reshape(n, 16, 16)
        return (w - (f16(82, 84)[:, None] * (sc >> 4))[:, :, None]).reshape(-1, K)
    q = (r[:, 32:96].reshape(n, 2, 1, 32) >> shift) & 3
    bit = torch.arange(8, device=raw.device, dtype=torch.int16).reshape(1, 2, 4, 1)
    q = q - 4 * (1 - ((r[:, :32].reshape(n, 1, 1, 32) >> bit) & 1))
    s = r[:, 96:108]
    i = torch.arange(16, device=raw.device)
    sc = ((s[:, i % 8] >> (4 * (i // 8)).short()) & 15) | (((s[:, 8 + i % 4] >> (2 * (i // 4)).short()) & 3) << 4)
    return ((f16(108, 110)[:, None] * (sc - 32))[:, :, None] * q.reshape(n, 16, 16)).reshape(-1, K)


def size_qs(fmt):
    return 16 if fmt == Q4 else 48


# ------------------------------------------------------------------------------------------------ a case's own data
def widths(case):
    return case["nh"] * case["hd"], case["nkv"] * case["hd"]


def layer_plan(case):
    """(name, rows, inputs) of one layer's matrices."""
    qd, kvd = widths(case)
    D, F = case["D"], case["F"]
    plan = []
    if case["kind"] != "moe":
        plan += [("q", qd, D), ("k", kvd, D), ("v", kvd, D), ("o", D, qd)]
    if F:
        plan += [("gate", F, D), ("up", F, D), ("down", D, F)]
    else:
        plan += [("eg", case["E"] * case["ffe"], D), ("eu", case["E"] * case["ffe"], D), ("ed", case["E"] * D, case["ffe"])]
    return plan


def ring(case, i):
    """(window, slots of the ring or 0, slots) of layer i: windows on all but the last layer."""
    swa = case.get("window", 0) if i < case["layers"] - 1 else 0
    cap = swa + case["batch"] if swa and case["ctx"] > swa + case["batch"] else 0
    return swa, cap, cap or case["ctx"]


def gen(case, seed):
    """Everything that the seed decides, as torch tensors on the GPU."""
    g = torch.Generator("cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    D, hd, T = case["D"], case["hd"], case["T"]
    _, kvd = widths(case)

    def norm(n):
        return 1.0 + 0.02 * torch.randn(n, generator=g, device="cuda")

    m = {"norm": norm(D), "layers": []}
    if case["kind"] == "sample":
        m["x"] = torch.randn(D, generator=g, device="cuda")
        m["out"] = gen_matrix(g, fmt_of(case, "out"), case["vocab"], D)
        m["pairs"] = torch.stack([torch.randperm(case["vocab"], generator=g, device="cuda")[:64].int(),
                                  torch.randint(1, 4, (64,), generator=g, device="cuda", dtype=torch.int32)], 1)
        return m
    rows = 4096
    m["emb"] = torch.randn(rows, D, generator=g, device="cuda")
    if case.get("window"):
        m["emb"] /= math.sqrt(D)   # these models scale their embeddings by sqrt(D)
    m["ids"] = torch.randint(0, rows, (T,), generator=g, device="cuda", dtype=torch.int32)
    if case["kind"] == "decode":
        m["out"] = gen_matrix(g, fmt_of(case, "out"), case["vocab"], D)
    for i in range(case["layers"]):
        L = {n: gen_matrix(g, fmt_of(case, n), N, K) for n, N, K in layer_plan(case)}
        L["attn_norm"], L["ffn_norm"] = norm(D), norm(D)
        if case["kind"] != "moe":
            if case.get("qk"):
                L["qnorm"], L["knorm"] = norm(hd), norm(hd)
            if case.get("window"):
                L["post_attn"], L["post_ffn"] = norm(D), norm(D)
            L["kc"] = torch.randn(case["pos"], kvd, generator=g, device="cuda")
            L["vc"] = torch.randn(case["pos"], kvd, generator=g, device="cuda")
            if case["f16"]:
                L["kc"], L["vc"] = L["kc"].half(), L["vc"].half()
        if not case["F"]:
            L["router"] = torch.randn(case["E"], D, generator=g, device="cuda") / math.sqrt(D)
        m["layers"].append(L)
    if case["kind"] == "moe" and case["used"] < case["E"]:
        # tokens whose last chosen and first rejected expert are not nearly tied (a tie is decided by rounding)
        L = m["layers"][0]
        lg = _rms(m["emb"].double(), L["ffn_norm"], 1e-6) @ L["router"].double().T
        top = lg.topk(case["used"] + 1, 1).values
        sure = ((top[:, -2] - top[:, -1]) > 1e-4).nonzero().reshape(-1)
        m["ids"] = sure[torch.randint(0, sure.numel(), (T,), generator=g, device="cuda")].int()
    return m


def eps_of(case):
    return 1e-6 if case.get("qk") or not case["F"] else 1e-5


def rope_base(case, i):
    if case.get("window"):
        return 10000.0 if i < case["layers"] - 1 else 1000000.0
    return 500000.0


def rope_table(base, hd):
    e = (np.float32(-2.0) * np.arange(hd // 2, dtype=np.float32)) / np.float32(hd)
    return np.power(float(base), e.astype(np.float64)).astype(np.float32)


# ------------------------------------------------------------------------------------------------- the user's program
_gpu = None


def gpu():
    global _gpu
    if _gpu is None:
        _gpu = capi.Quipu(0)
    return _gpu


class Memory:
    """A part of a buffer as torch takes it; the tensor holds on to it, and it to the buffer."""

    def __init__(self, buffer, shape, typestr, offset):
        self.buffer = buffer
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "version": 2, "strides": None,
                                         "data": (buffer.h + offset, False)}


class Buffer:
    """A buffer of the library, freed with its last reference."""

    def __init__(self, nbytes, data=None, zero=False):
        self.n = max(16, (int(nbytes) + 3) // 4 * 4)
        self.h = gpu().alloc(self.n)
        if zero:
            gpu().dispatch("fill_u32", [("u", 0), ("u", self.n // 4), ("u", 0)], [0, self.h])
        if data is not None:
            data = data.contiguous()
            torch.cuda.current_stream().synchronize()
            gpu().copy(self.h, data.data_ptr(), data.numel() * data.element_size())
            gpu().sync()

    def __del__(self):
        gpu().free(self.h)

    def view(self, shape, typestr="<f4", offset=0):
        """The buffer's memory as a torch tensor (no copy)."""
        return torch.as_tensor(Memory(self, shape, typestr, offset), device="cuda")


class Plan:
    """Dispatches with their uniforms and bindings packed once (the engine's bind groups)."""

    def __init__(self):
        self.calls = []

    def add(self, op, u, bufs, grid=(1, 1, 1)):
        ub = capi.uniform(u)
        hs = [b.h if isinstance(b, Buffer) else int(b or 0) for b in bufs]
        grid = tuple(grid) + (1,) * (3 - len(grid))
        self.calls.append((gpu().op(op), ctypes.create_string_buffer(ub, len(ub)), len(ub),
                           (ctypes.c_uint64 * len(hs))(*hs), len(hs)) + grid)

    def run(self):
        dispatch = gpu().L.qp_dispatch
        for c in self.calls:
            if dispatch(*c):
                gpu()._check(1, "qp_dispatch")


class Matrix:
    def __init__(self, raw, fmt, N, K):
        self.fmt, self.N, self.K, self.name = fmt, N, K, NAME[fmt]
        if fmt == F32:
            self.buf = Buffer(4 * N * K, raw)
        else:
            src = Buffer(raw.numel(), raw)
            self.buf = Buffer(capi.device_bytes(fmt, N, K))
            nb = raw.shape[0]
            gpu().dispatch("repack_" + self.name, [("u", nb & 0xFFFFFFFF), ("u", nb >> 32), ("u", K)], [0, src.h, self.buf.h])
            gpu().sync()
        self.w = [self.buf.h]
        if fmt in PLANAR:
            self.w.append(capi.scale_plane(fmt, self.buf.h, N, K))


def f32(t):
    return Buffer(4 * t.numel(), t.float())


def v_tiles(v):
    """The f16 value cache's layout: tiles of 32 slots, per channel the slots in the order 8 (k % 16 / 4) + 4 (k / 16)
    + k % 4."""
    pad = -v.shape[0] % 32
    t = torch.nn.functional.pad(v, (0, 0, 0, pad)).reshape(-1, 32, v.shape[1])
    k = torch.arange(32, device=v.device)
    out = torch.empty_like(t)
    out[:, 8 * ((k % 16) // 4) + 4 * (k // 16) + k % 4] = t
    return out.transpose(1, 2).contiguous()


class State:
    """The model, buffers and dispatch plan that a program keeps, built as the engine's model class builds them."""

    graph = None

    def __init__(self, case, seed):
        self.case = case
        m = gen(case, seed)
        self.m = {"norm": f32(m["norm"])}
        self.plan = Plan()
        T, D = case["T"], case["D"]
        self.paso = Buffer(16)
        gpu().upload(self.paso.h, np.array([T, case.get("pos", 0), 0, 0], np.uint32))
        self.keep = []
        self.x = Buffer(4 * T * D)
        if case["kind"] == "sample":
            self._sample(m)
            return
        self.m["emb"] = f32(m["emb"])
        self.ids = Buffer(4 * T, m["ids"])
        self.layers = [self._layer(m["layers"][i], i) for i in range(case["layers"])]
        for L in m["layers"]:
            L.clear()
        if case["kind"] == "decode":
            self.out = Matrix(m["out"], fmt_of(case, "out"), case["vocab"], D)
            self._decode()
        else:
            self._prefill()

    def __del__(self):
        if self.graph:
            gpu().sync()
            gpu().graph_free(self.graph)

    def new(self, nbytes, zero=False):
        b = Buffer(nbytes, zero=zero)
        self.keep.append(b)
        return b

    def _layer(self, raw, i):
        c = self.case
        L = {n: Matrix(raw[n], fmt_of(c, n), N, K) for n, N, K in layer_plan(c)}
        for n in ("attn_norm", "ffn_norm", "qnorm", "knorm", "post_attn", "post_ffn"):
            L[n] = f32(raw[n]) if n in raw else None
        if "router" in raw:
            L["router"] = Matrix(raw["router"].reshape(-1, 1).view(torch.uint8), F32, c["E"], c["D"])
        if "kc" in raw:
            kvd = widths(c)[1]
            L["swa"], L["cap"], L["slots"] = ring(c, i)
            slots, kind = L["slots"], torch.float16 if c["f16"] else torch.float32
            K, V = (torch.zeros(slots, kvd, dtype=kind, device="cuda") for _ in range(2))
            p = torch.arange(max(0, c["pos"] - slots), c["pos"], device="cuda")
            K[p % slots], V[p % slots] = raw["kc"][p], raw["vc"][p]
            if c["f16"]:
                V = v_tiles(V)
            L["kc"], L["vc"] = (Buffer(t.numel() * t.element_size(), t) for t in (K, V))
            L["base"] = rope_base(c, i)
            L["freq"] = Buffer(2 * c["hd"], torch.from_numpy(rope_table(L["base"], c["hd"])))
        return L

    # ---- prompt chunks, op by op
    def _mm(self, W, x, y, acc=0, mode=0, one=None):
        T, add = self.case["T"], self.plan.add
        u = [("u", W.N), ("u", W.K), ("u", acc), ("u", 0)]
        b = [self.paso] + W.w + [x, y]
        if T == 1 or one:
            add("matmul_%s_1" % W.name, u, b, capi.dim2((W.N + 7) // 8))
        elif T >= 8 and W.fmt in KQ:
            add("matmul_%s_t" % W.name, u + ([("u", mode)] if mode else []), b, ((W.N + 63) // 64, 1, (T + 31) // 32))
        else:
            add("matmul_%s_4" % W.name, u, b, capi.dim2((W.N + 7) // 8) + ((T + 3) // 4,))

    def _prefill(self):
        c, add, P = self.case, self.plan.add, self.paso
        T, D, hd, nh, nkv, F = c["T"], c["D"], c["hd"], c["nh"], c["nkv"], c["F"]
        qd, kvd = widths(c)
        eps, window = eps_of(c), c.get("window", 0)
        neox = 1 if c.get("qk") else 0
        rows = lambda n: ((T * n + 255) // 256,)   # noqa: E731
        T256 = (T + 255) // 256 * 256
        big = T >= 256 and not window
        xn = self.new(4 * T * max(D, 1))
        add("embed_f32", [("u", D), ("u", 4096)], [P, self.m["emb"], self.ids, self.x], rows(D))
        if window:
            add("escalar", [("u", D), ("f", math.sqrt(D))], [P, self.x], rows(D))
        planes = self.new(4 * T256 * max(D, qd)) if big else None
        tmp = self.new(4 * T * D) if window else None
        if c["kind"] != "moe":
            q, k, v, att = self.new(4 * T * qd), self.new(4 * T * kvd), self.new(4 * T * kvd), self.new(4 * T * qd)
            self.k = k
        if F:
            g, u = self.new(4 * T256 * F), self.new(4 * T * F)
        u_norm = [("u", D), ("u", 0), ("f", eps), ("u", 0)]

        def residual(W, x, post, mode=0):
            if not post:
                self._mm(W, x, self.x, 1, mode)
                return
            self._mm(W, x, tmp, 0, mode)
            add("rmsnorm", u_norm, [P, tmp, post, xn], (T,))
            add("suma_esc", [("u", D), ("f", 1.0)], [P, self.x, xn], rows(D))

        for L in self.layers:
            if c["kind"] != "moe":
                self._attention(L, xn, q, k, v, att, planes, u_norm, residual, neox, big)
            if not F:
                self._experts(L, xn, u_norm)
                continue
            glu = big and L["gate"].fmt in KQ
            if glu:
                add("rmsnorm_planes", [("u", D), ("f", eps)], [P, self.x, L["ffn_norm"], planes], ((T + 7) // 8,))
                yp = 1 if L["down"].fmt in KQ else 0
                add("matmul_%s_t_swiglu" % L["gate"].name, [("u", F), ("u", D), ("u", yp), ("u", 1)],
                    [P] + L["gate"].w + L["up"].w + [planes, g], ((F + 63) // 64, 1, (T + 31) // 32))
                residual(L["down"], g, L["post_ffn"], 2 if yp else 0)
            else:
                add("rmsnorm", u_norm, [P, self.x, L["ffn_norm"], xn], (T,))
                self._mm(L["gate"], xn, g)
                self._mm(L["up"], xn, u)
                add("geglu" if window else "swiglu", [("u", F)], [P, g, u], rows(F))
                residual(L["down"], g, L["post_ffn"])

    def _attention(self, L, xn, q, k, v, att, planes, u_norm, residual, neox, big):
        c, add, P = self.case, self.plan.add, self.paso
        T, D, hd, nh, nkv = c["T"], c["D"], c["hd"], c["nh"], c["nkv"]
        qd, kvd = widths(c)
        eps = eps_of(c)
        if big and all(L[n].fmt in KQ for n in "qkv"):
            add("rmsnorm_planes", [("u", D), ("f", eps)], [P, self.x, L["attn_norm"], planes], ((T + 7) // 8,))
            for n, y in (("q", q), ("k", k), ("v", v)):
                self._mm(L[n], planes, y, 0, 2)
        else:
            add("rmsnorm", u_norm, [P, self.x, L["attn_norm"], xn], (T,))
            reuse = 0 if c.get("window") else 1
            for n, y, mode in (("q", q, 0), ("k", k, reuse), ("v", v, reuse)):
                self._mm(L[n], xn, y, 0, mode)
        for y, heads, norm in ((q, nh, L["qnorm"]), (k, nkv, L["knorm"])):
            add("norm_rope", [("u", hd), ("u", heads), ("u", 1 if norm else 0), ("u", neox), ("f", eps),
                              ("f", L["base"]), ("u", hd), ("f", 0.0)], [P, y, norm or self.m["norm"], L["freq"]], (heads, T))
        add("kv_write", [("u", kvd), ("u", L["cap"]), ("u", c["f16"]), ("u", L["slots"])], [P, k, v, L["kc"], L["vc"]],
            ((T * kvd + 255) // 256,))
        u_att = [("u", hd), ("u", nh), ("u", nkv), ("u", L["swa"]), ("f", 1.0 / math.sqrt(hd)), ("u", L["cap"]), ("u", 0),
                 ("u", 0), ("u", c["f16"]), ("u", L["slots"])]
        if big and L["o"].fmt in KQ and c["f16"] and not L["swa"]:
            add("atencion", u_att + [("u", 1)], [P, q, L["kc"], L["vc"], planes], (nh, T))
            residual(L["o"], planes, L["post_attn"], 2)
        else:
            add("atencion", u_att, [P, q, L["kc"], L["vc"], att], (nh, T))
            residual(L["o"], att, L["post_attn"])

    def _experts(self, L, xn, u_norm):
        c, add, P = self.case, self.plan.add, self.paso
        T, D, E, used, ffe = c["T"], c["D"], c["E"], c["used"], c["ffe"]
        rl, sel, wts = self.new(4 * T * E), self.new(4 * T * used), self.new(4 * T * used)
        lst, off = self.new(4 * T * used), self.new(4 * (E + 1))
        g, u, de = self.new(4 * T * used * ffe), self.new(4 * T * used * ffe), self.new(4 * T * used * D)
        add("rmsnorm", u_norm, [P, self.x, L["ffn_norm"], xn], (T,))
        self._mm(L["router"], xn, rl)
        add("moe_topk", [("u", E), ("u", used), ("u", 1), ("f", 1.0)], [P, rl, sel, wts], ((T + 63) // 64,))
        if T >= 8:
            add("moe_group", [("u", E), ("u", used)], [P, sel, lst, off])

        def expert(W, x, y, fixed, per_token, reuse):
            n = W.N // E
            if T >= 8:
                add("matmul_%s_eg" % W.name, [("u", n), ("u", W.K), ("u", 0), ("u", fixed), ("u", per_token), ("u", reuse)],
                    [P] + W.w + [x, y, lst, off], ((n + 63) // 64, E, (T + 31) // 32))
            else:
                add("matmul_%s_e" % W.name, [("u", n), ("u", W.K), ("u", 0), ("u", fixed), ("u", E)],
                    [P] + W.w + [x, y, sel], capi.dim2((n + 7) // 8) + (T * used,))

        expert(L["eg"], xn, g, used, 1, 0)
        expert(L["eu"], xn, u, used, 1, 1)
        add("swiglu", [("u", used * ffe)], [P, g, u], ((T * used * ffe + 255) // 256,))
        expert(L["ed"], g, de, 1, used, 0)
        add("moe_comb", [("u", D), ("u", used)], [P, self.x, de, wts], ((T * D + 255) // 256,))

    # ---- one token, fused and captured
    def _gemv(self, segs, x, norm, K, R=0, max_wg=0, amax=0):
        f = segs[0][0].fmt
        u = capi.gemv_uniform(len(segs), K, eps=eps_of(self.case), R=R, max_wg=max_wg, fmt=f,
                              segs=[(mode, W.N, 0, W.N, W.fmt if W.fmt != f else 0) for W, _, mode, _ in segs])
        b = [self.paso, x, norm or 0, amax]
        for W, W2, _, y in segs:
            b += [W.w[0], W2.w[0] if W2 else 0, y]
        self.plan.add("gemv", u, b)

    def _gemv_by_format(self, segs, x, norm, K):
        groups = {}
        for s in segs:
            groups.setdefault("kq" if s[0].fmt in MIXED else s[0].fmt, []).append(s)
        for g in groups.values():
            self._gemv(g, x, norm, K)

    def _decode(self):
        c, add, P = self.case, self.plan.add, self.paso
        D, hd, nh, nkv, F = c["D"], c["hd"], c["nh"], c["nkv"], c["F"]
        qd, kvd = widths(c)
        eps = eps_of(c)
        neox = 1 if c.get("qk") else 0
        q, k, v, att = self.new(4 * qd), self.new(4 * kvd), self.new(4 * kvd), self.new(4 * qd)
        per = 256 if nkv * -(-c["ctx"] // 256) >= 64 else 128
        ns = max(1, min(256, -(-c["ctx"] // per)))
        part_o, part_ml = self.new(4 * nh * ns * hd), self.new(8 * nh * ns)
        counters = self.new(8 * 128 + 128, zero=True)
        group, split = nh // nkv, 1
        while group // split > 4 and split < 8:
            split *= 2
        merged = nkv * split <= 8 and group % split == 0 and group // split <= 4
        add("embed_f32", [("u", D), ("u", 4096)], [P, self.m["emb"], self.ids, self.x], ((D + 255) // 256,))
        for L in self.layers:
            self._gemv_by_format([(L["q"], None, STORE, q), (L["k"], None, STORE, k), (L["v"], None, STORE, v)], self.x,
                                 L["attn_norm"], D)
            u = [("u", hd), ("u", nh), ("u", nkv), ("u", ns), ("f", 1.0 / math.sqrt(hd)), ("f", eps), ("f", L["base"]),
                 ("u", 0), ("u", hd), ("u", neox), ("u", c["f16"]), ("u", c["ctx"])]
            b = [P, q, k, v, L["kc"], L["vc"], L["qnorm"] or 0, L["knorm"] or 0, part_o, part_ml, L["freq"]]
            if merged:
                add("dec_attn", u + [("u", 1), ("u", split)], b + [att, counters])
            else:
                add("dec_attn", u, b)
                add("dec_attn_comb", [("u", hd), ("u", nh), ("u", ns)], [P, part_o, part_ml, att])
            self._gemv([(L["o"], None, ACC, self.x)], att, None, qd)
            if F:
                g = self.new(4 * F)
                self._gemv([(L["gate"], L["up"], SWIGLU, g)], self.x, L["ffn_norm"], D)
                self._gemv([(L["down"], None, ACC, self.x)], g, None, F)
            else:
                E, used, ffe = c["E"], c["used"], c["ffe"]
                rl, sel, wts, cnt = self.new(4 * E), self.new(4 * used), self.new(4 * used), self.new(8, zero=True)
                g = self.new(4 * used * ffe)
                nw = 1
                while nw * 4 < E and nw * 2 <= 64:
                    nw *= 2
                add("moe_router", [("u", E), ("u", D), ("u", used), ("u", nw), ("f", eps), ("f", 1.0), ("u", 1)],
                    [P] + L["router"].w + [self.x, L["ffn_norm"], rl, sel, wts, cnt])
                add("moe_gate_up_" + L["eg"].name, [("u", ffe), ("u", D), ("u", E), ("u", used), ("f", eps), ("f", 1.0),
                                                    ("u", 1), ("u", 1)],
                    [P] + L["eg"].w + L["eu"].w + [self.x, L["ffn_norm"], rl, g, sel, wts])
                add("moe_down_" + L["ed"].name, [("u", D), ("u", ffe), ("u", E), ("u", used), ("f", eps), ("f", 1.0),
                                                 ("u", 1)], [P] + L["ed"].w + [g, self.x, sel, wts])
        self._head()
        self.plan.run()   # once eagerly, then captured, as the engine does
        gpu().sync()
        gpu().graph_begin()
        self.plan.run()
        self.graph = gpu().graph_end()
        gpu().sync()

    def _head(self):
        c = self.case
        V = c["vocab"]
        self.logits, self.token = Buffer(4 * V), Buffer(16)
        r = 2 if self.out.fmt == Q6 else 4
        wg = min(512, -(-V // (4 * r)))
        amax, step = self.new(8 * 512, zero=True), self.new(16, zero=True)
        self._gemv([(self.out, None, ARGMAX, self.logits)], self.x, self.m["norm"], c["D"], R=r, max_wg=wg, amax=amax)
        self.plan.add("argmax_fin", [("u", wg), ("u", 0), ("u", 0)], [self.paso, amax, self.token, 0, step])

    # ---- output matrix, penalties, candidates
    def _sample(self, m):
        c, add = self.case, self.plan.add
        V, k = c["vocab"], c["topk"]
        self.x = f32(m["x"])
        self.out = Matrix(m["out"], fmt_of(c, "out"), V, c["D"])
        self._head()
        pairs = Buffer(512, m["pairs"])
        self.keep.append(pairs)
        u = [("u", 64), ("u", V)]
        for f in (1.1, 0.0, 0.0):
            bits = int(np.float64(f).view(np.uint64))
            u += [("u", bits & 0xFFFFFFFF), ("u", bits >> 32)]
        chunks = -(-V // 2048)
        part, self.cand = self.new(chunks * (k + 1) * 8 + chunks * 4), Buffer(4 * (2 + 2 * k))
        add("penalizar", u, [self.logits, pairs])
        add("topk_cand", [("u", V), ("u", k)], [self.logits, part, self.cand])

    def run(self):
        if self.graph:
            gpu().graph_launch(self.graph)
        else:
            self.plan.run()
        return self.outputs

    def make_outputs(self):
        c = self.case
        if c["kind"] == "sample":
            cand = self.cand.view((1 + c["topk"], 2))
            self.outputs = {"logits": self.logits.view((c["vocab"],)), "values": cand[1:, 0]}
        elif c["kind"] == "decode":
            kvd, size, typ = widths(c)[1], 2 if c["f16"] else 4, "<f2" if c["f16"] else "<f4"
            self.outputs = {"logits": self.logits.view((c["vocab"],)), "token": self.token.view((1,), "<i4"),
                            "x": self.x.view((c["D"],)),
                            "keys": [L["kc"].view((kvd,), typ, c["pos"] * kvd * size) for L in self.layers]}
        else:
            self.outputs = {"x": self.x.view((c["T"], c["D"]))}
            if c["kind"] != "moe":
                self.outputs["k"] = self.k.view((c["T"], widths(c)[1]))


def prepare(case, seed):
    s = State(case, seed)
    s.make_outputs()
    return s


def run(state):
    return state.run()


# ------------------------------------------------------------------------------------------------ what it comes down to
def work(case):
    T, D = case["T"], case["D"]
    per, flops, byts = lambda f: _BYTES[f][1] / _BYTES[f][0], 0.0, 0.0   # noqa: E731
    qd, kvd = widths(case)
    if case["kind"] in ("decode", "sample"):
        n = case["vocab"] * D
        flops += 2.0 * n
        byts += n * per(fmt_of(case, "out")) + 4.0 * case["vocab"]
    if case["kind"] != "sample":
        byts += 8.0 * T * D    # embedding rows in, activations out
        for i in range(case["layers"]):
            for n, N, K in layer_plan(case):
                if n[0] == "e":
                    E, used = case["E"], case["used"]
                    flops += 2.0 * T * used * (N // E) * K
                    byts += N * K * per(fmt_of(case, n)) * (1.0 - (1.0 - used / E) ** T)
                else:
                    flops += 2.0 * T * N * K
                    byts += N * K * per(fmt_of(case, n))
            if not case["F"]:
                flops += 2.0 * T * case["E"] * D
                byts += 4.0 * case["E"] * D
            if case["kind"] != "moe":
                swa = ring(dict(case, batch=case.get("batch", 1)), i)[0]
                keys = [min(case["pos"] + t + 1, swa or 1 << 30) for t in (0, T - 1)]
                flops += 4.0 * T * (keys[0] + keys[1]) / 2 * qd
                byts += 2.0 * (2 if case["f16"] else 4) * kvd * (min(case["pos"], swa or 1 << 30) + T)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """About four times what the path differs by from `exact`: 32-bit sums through one to eight layers (1e-7 to 4e-7),
    matrix-core products that keep about 16 bits of each factor (2e-6 to 1.4e-5 from 64 tokens on), and with the f16 cache
    a key or value now and then rounded to the neighbouring half (1e-5 to 8e-5 of a step's few keys)."""
    if case["kind"] == "sample":
        return {"rel": 1e-6}
    if case["kind"] == "moe":
        return {"rel": 1e-5}
    if case["kind"] == "decode":
        return {"rel": 3e-4, "max": 4e-3} if case["f16"] else {"rel": 2e-6}
    return {"rel": 6e-5, "max": 4e-3}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _lin(raw, fmt, K, x):
    """x W^T, some rows of W at a time."""
    blocks = K // _BYTES[fmt][0]
    rows = max(1, (1 << 26) // K)
    return torch.cat([x @ dequant(raw[a:a + rows * blocks], fmt, K).T for a in range(0, raw.shape[0], rows * blocks)], -1)


def _rope(v, pos, base, neox):
    """v [T, heads, hd]; the angle is the 32-bit product of position and table entry, as everywhere in this family."""
    hd = v.shape[-1]
    f = torch.from_numpy(rope_table(base, hd)).cuda()
    th = (pos.float()[:, None] * f[None]).double()[:, None, :]
    a, b = (v[..., :hd // 2], v[..., hd // 2:]) if neox else (v[..., 0::2], v[..., 1::2])
    r = (a * th.cos() - b * th.sin(), a * th.sin() + b * th.cos())
    return torch.cat(r, -1) if neox else torch.stack(r, -1).flatten(-2)


def _attend(q, k, v, pos, swa, scale):
    """q [T, nh, hd] at positions pos over k, v [n, nkv, hd]; a head at a time."""
    n, out = k.shape[0], torch.empty_like(q)
    j = torch.arange(n, device=q.device)
    hidden = j[None] > pos[:, None]
    if swa:
        hidden |= j[None] <= pos[:, None] - swa
    g = q.shape[1] // k.shape[1]
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // g].T) * scale
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, h // g]
    return out


def exact(case, seed):
    m = gen(case, seed)
    c, D, eps = case, case["D"], eps_of(case)
    if c["kind"] == "sample":
        lg = _lin(m["out"], fmt_of(c, "out"), D, _rms(m["x"].double(), m["norm"], eps))
        t = m["pairs"][:, 0].long()
        lg[t] = torch.where(lg[t] > 0, lg[t] / 1.1, lg[t] * 1.1)
        return {"logits": lg, "values": lg.topk(c["topk"]).values}
    T, hd, nh, nkv, window = c["T"], c["hd"], c["nh"], c["nkv"], c.get("window", 0)
    x = m["emb"][m["ids"].long()].double()
    if window:
        x = x * math.sqrt(D)
    pos = torch.arange(T, device="cuda") + c.get("pos", 0)
    keys = []
    for i, L in enumerate(m["layers"]):
        if c["kind"] != "moe":
            xn = _rms(x, L["attn_norm"], eps)
            q, k, v = (_lin(L[n], fmt_of(c, n), D, xn).reshape(T, -1, hd) for n in "qkv")
            if c.get("qk"):
                q, k = _rms(q, L["qnorm"], eps), _rms(k, L["knorm"], eps)
            q, k = (_rope(y, pos, rope_base(c, i), bool(c.get("qk"))) for y in (q, k))
            keys.append(k.reshape(T, -1))
            if c["f16"]:
                k, v = k.half().double(), v.half().double()
            if c["kind"] == "decode":
                keys[-1] = k.reshape(-1)
            k = torch.cat([L["kc"].double().reshape(-1, nkv, hd), k])
            v = torch.cat([L["vc"].double().reshape(-1, nkv, hd), v])
            o = _attend(q, k, v, pos, ring(dict(c, batch=c.get("batch", 1)), i)[0], 1.0 / math.sqrt(hd))
            o = _lin(L["o"], fmt_of(c, "o"), nh * hd, o.reshape(T, -1))
            x = x + (_rms(o, L["post_attn"], eps) if window else o)
        xn = _rms(x, L["ffn_norm"], eps)
        if c["F"]:
            g, u = (_lin(L[n], fmt_of(c, n), D, xn) for n in ("gate", "up"))
            h = torch.nn.functional.gelu(g, approximate="tanh") * u if window else torch.nn.functional.silu(g) * u
            o = _lin(L["down"], fmt_of(c, "down"), c["F"], h)
            x = x + (_rms(o, L["post_ffn"], eps) if window else o)
        else:
            E, used, ffe = c["E"], c["used"], c["ffe"]
            top = (xn @ L["router"].double().T).softmax(-1).topk(used, -1)
            w = top.values / top.values.sum(-1, keepdim=True)
            o = torch.zeros_like(x)
            for e in range(E):
                t, s = (top.indices == e).nonzero(as_tuple=True)
                if t.numel():
                    part = lambda n, N, K: L[n].reshape(E, -1, L[n].shape[-1])[e]   # noqa: E731
                    g, u = (_lin(part(n, ffe, D), fmt_of(c, n), D, xn[t]) for n in ("eg", "eu"))
                    y = _lin(part("ed", D, ffe), fmt_of(c, "ed"), ffe, torch.nn.functional.silu(g) * u)
                    o.index_add_(0, t, y * w[t, s][:, None])
            x = x + o
    if c["kind"] == "decode":
        lg = _lin(m["out"], fmt_of(c, "out"), D, _rms(x, m["norm"], eps)).reshape(-1)
        return {"logits": lg, "token": None, "x": x.reshape(-1), "keys": keys}
    return {"x": x, "k": keys[-1]} if c["kind"] != "moe" else {"x": x}
