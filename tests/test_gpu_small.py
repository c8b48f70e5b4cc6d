"""The integer-weight matmuls of few token rows (qp_small.hip) against float64, at the edges of their tiles.

Bound: the weights are exact and x keeps 22 bits below its largest magnitude per 256 inputs, so what is left is the
rounding of float32 sums.  An output adds at most A = K / 16 + K / 64 terms in a row (two or three matrix instructions
per 32 inputs, each adding to the running sum; one addition per 256 inputs and K slice), each rounding to 2^-24 of a
partial sum of at most S = sum |x_k| (|scale * quant| + |minimum|); roundings of either sign make sqrt(A) of them count.
The test allows 4 sqrt(A) 2^-24 S.  S is at most 3 sum |x_k| max |w| for these random blocks' rows (quants of the whole
range, minima no larger than the largest product).
"""
import numpy as np
import pytest

from quipullm_amd import capi
from test_gpu_ops import FMTS, PLANAR, dev, raw_matrix, topk_cand  # noqa: F401

pytestmark = pytest.mark.gpu


def weights(oracle, fmt, raw, N, K):
    return (oracle.dequant(fmt, raw, N * K) if fmt != capi.F32 else raw.view(np.float32)).reshape(N, K).astype(np.float64)


def bound(W, x):
    K = W.shape[1]
    return 4 * np.sqrt(K / 16 + K / 64) * 2.0 ** -24 * 3 * np.abs(x.astype(np.float64)).sum(1)[:, None] * np.abs(W).max(1)[None]


def matmul(quipu, dev, fmt, raw, N, K, x, y0=None, t_op=True):
    T = x.shape[0]
    y = dev.buf(np.full((T + 2, N), 7.0, np.float32) if y0 is None else np.vstack([y0, np.full((2, N), 7.0, np.float32)]))
    wb = [dev.matrix(fmt, raw, N, K)]
    if fmt in PLANAR:
        wb.append(capi.scale_plane(fmt, wb[0], N, K))
    grid = ((N + 63) // 64, 1, (T + 31) // 32) if t_op else capi.dim2((N + 7) // 8) + ((T + 3) // 4,)
    quipu.dispatch("matmul_%s_%s" % (capi.FMT_NAME[fmt], "t" if t_op else "4"),
                   [("u", N), ("u", K), ("u", y0 is not None), ("u", 0)], [dev.paso(T, 0)] + wb + [dev.buf(x), y], grid)
    out = dev.get(y, (T + 2, N))
    assert np.all(out[T:] == 7.0)  # rows past T are not written
    return out[:T]


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("T,N,K", [(2, 1, 256), (15, 17, 768), (17, 200, 1280), (33, 33, 2048), (64, 130, 4352),
                                   (65, 16, 1024), (130, 4100, 512), (255, 96, 5376)])
def test_few_tokens(quipu, dev, oracle, fmt, T, N, K):
    """Tile and block edges: one row, 16 and 16 + 1 rows, token tiles of 16, 32 and 64 with remainders, K of one block, of
    part of a group of four, and of more groups than K slices."""
    raw = raw_matrix(fmt, N, K, 71)
    W = weights(oracle, fmt, raw, N, K)
    rng = np.random.default_rng(72)
    x = rng.standard_normal((T, K)).astype(np.float32)
    y0 = rng.standard_normal((T, N)).astype(np.float32) if T % 2 else None
    got = matmul(quipu, dev, fmt, raw, N, K, x, y0, t_op=T % 3 != 0)
    want = x.astype(np.float64) @ W.T + (0 if y0 is None else y0)
    assert np.all(np.abs(got - want) <= bound(W, x) + (0 if y0 is None else 2.0 ** -23 * np.abs(y0)))


@pytest.mark.parametrize("fmt,K", [(capi.Q8_0, 32), (capi.Q8_0, 288), (capi.IQ4_NL, 96), (capi.IQ4_NL, 544),
                                   (capi.F32, 16), (capi.F32, 272), (capi.F32, 1040)])
def test_few_tokens_ragged_k(quipu, dev, oracle, fmt, K):
    """K that is no multiple of 256: the last chunk's missing blocks are zeros on both sides."""
    T, N = 19, 37
    raw = raw_matrix(fmt, N, K, 73)
    W = weights(oracle, fmt, raw, N, K)
    x = np.random.default_rng(74).standard_normal((T, K)).astype(np.float32)
    assert np.all(np.abs(matmul(quipu, dev, fmt, raw, N, K, x, t_op=False) - x.astype(np.float64) @ W.T) <= bound(W, x))


@pytest.mark.parametrize("fmt", [capi.Q4_K, capi.Q6_K, capi.Q8_0, capi.F32])
def test_few_tokens_magnitudes(quipu, dev, oracle, fmt):
    """Rows of magnitude 1e-30 .. 1e30, a zero row, a row of denormals, an outlier, and rows with an infinity and a NaN,
    which stay in their own rows."""
    T, N, K = 40, 50, 1024
    raw = raw_matrix(fmt, N, K, 75)
    W = weights(oracle, fmt, raw, N, K)
    rng = np.random.default_rng(76)
    x = (rng.standard_normal((T, K)) * 10.0 ** rng.integers(-30, 31, size=T)[:, None]).astype(np.float32)
    x[3] = 0.0
    x[4] = (rng.standard_normal(K) * 1e-39).astype(np.float32)
    x[5, 7] *= 1e6
    x[6, 100] = np.inf
    x[7, 300] = np.nan
    got = matmul(quipu, dev, fmt, raw, N, K, x)
    ok = [t for t in range(T) if t not in (6, 7)]
    want = x[ok].astype(np.float64) @ W.T
    assert np.all(got[3] == 0.0) and not np.isfinite(got[[6, 7]]).any()
    assert np.all(np.abs(got[ok] - want) <= bound(W, x[ok]) + 1e-37)  # (sums below the smallest normal may be flushed)


@pytest.mark.parametrize("fmt", FMTS)
def test_few_jobs_per_expert(quipu, dev, oracle, fmt):
    """matmul_<fmt>_eg with few jobs per expert: experts without jobs, one with every token (more than a tile), gathered
    input rows (tfijo = 3) and job rows; the two of them with and without P[4] give the same bits."""
    E, N, K, k, T = 9, 70, 768, 3, 21
    rng = np.random.default_rng(77)
    sel = np.stack([np.concatenate([[4], rng.choice([0, 2, 7], 2, replace=False)]) for _ in range(T)]).astype(np.uint32).ravel()
    raw = raw_matrix(fmt, E * N, K, 78)
    W = weights(oracle, fmt, raw, E * N, K).reshape(E, N, K)
    hw = dev.matrix(fmt, raw, E * N, K)
    wb = [hw, capi.scale_plane(fmt, hw, E * N, K)] if fmt in PLANAR else [hw]
    sb, lb, ob = dev.buf(sel), dev.zeros(4 * T * k), dev.zeros(4 * (E + 1))
    p = dev.paso(T, 0)
    quipu.dispatch("moe_group", [("u", E), ("u", k)], [p, sb, lb, ob])
    for tfijo, m in ((k, 1), (1, k)):
        x = rng.standard_normal((T * k // tfijo, K)).astype(np.float32)
        xb, outs = dev.buf(x), []
        for extra in ([("u", m), ("u", 0)], []):
            y = dev.zeros(4 * T * k * N)
            quipu.dispatch("matmul_%s_eg" % capi.FMT_NAME[fmt], [("u", N), ("u", K), ("u", 0), ("u", tfijo)] + extra,
                           [p] + wb + [xb, y, lb, ob], ((N + 63) // 64, E, 1))
            outs.append(dev.get(y, (T * k, N)))
        assert np.array_equal(outs[0], outs[1])
        for j in range(T * k):
            e = sel[j]
            xr = x[j // tfijo][None]
            assert np.all(np.abs(outs[0][j] - (xr.astype(np.float64) @ W[e].T)[0]) <= bound(W[e], xr)[0]), j


def split_bound(W, x):
    """x read as its bfloat16 high + low parts, each input off by at most 2^-18 of itself, roundings of either sign."""
    return bound(W, x) + 4 * 2.0 ** -18 * np.sqrt(x.astype(np.float64) ** 2 @ (W ** 2).T)


KQ = [f for f in FMTS if f not in PLANAR and f != capi.F32]


@pytest.mark.parametrize("fmt", KQ)
@pytest.mark.parametrize("T,N,K", [
    (256, 128, 256), (257, 1, 512), (321, 129, 768), (383, 250, 1280), (512, 512, 4096), (1000, 768, 2048),  # few workgroups
    (2176, 1152, 256), (2049, 1100, 512), (577, 129, 3328), (513, 1, 4352), (832, 250, 5376)])               # 128 x 128 tiles
def test_many_tokens(quipu, dev, oracle, fmt, T, N, K):
    """256 tokens and more.  Matrices of so few workgroups that each wavefront keeps its weights (up to exactly a workgroup
    per CU of 256): one block of 256 inputs to four K slices, one row, remainders.  The 128 x 128 tiles: whole ones, one row,
    one token and one row past a tile, a tile of 64 tokens, one block of 256 inputs, K splits with a shorter last one."""
    raw = raw_matrix(fmt, N, K, 81)
    W = weights(oracle, fmt, raw, N, K)
    rng = np.random.default_rng(82)
    x = rng.standard_normal((T, K)).astype(np.float32)
    y0 = rng.standard_normal((T, N)).astype(np.float32) if T % 2 else None
    got = matmul(quipu, dev, fmt, raw, N, K, x, y0)
    want = x.astype(np.float64) @ W.T + (0 if y0 is None else y0)
    assert np.all(np.abs(got - want) <= split_bound(W, x) + (0 if y0 is None else 2.0 ** -23 * np.abs(y0)))


@pytest.mark.parametrize("T,N,K", [(513, 1000, 10240), (640, 2000, 8192), (1100, 2000, 8192), (130, 8200, 8192)])
def test_k_splits_on_their_xcds(quipu, dev, oracle, T, N, K):
    """Q6_K tiles of long rows in 8, 4, 2 and 2 K splits, each on its share of the XCDs, tiles that do not divide by it."""
    test_many_tokens(quipu, dev, oracle, capi.Q6_K, T, N, K)


@pytest.mark.parametrize("fmt", KQ)
@pytest.mark.parametrize("T,N,K", [(256, 64, 256), (300, 97, 768), (390, 200, 512)])
def test_many_tokens_swiglu(quipu, dev, oracle, fmt, T, N, K):
    """matmul_<fmt>_t_swiglu: silu(g) u of the two products; |silu'| < 1.1, and 2^-20 for the exponential, the division and
    the product."""
    raw = [raw_matrix(fmt, N, K, 83 + i) for i in range(2)]
    W = [weights(oracle, fmt, r, N, K) for r in raw]
    x = (np.random.default_rng(85).standard_normal((T, K)) / np.sqrt(K) / np.abs(W[0]).max()).astype(np.float32)
    y = dev.buf(np.full((T + 1, N), 7.0, np.float32))
    quipu.dispatch("matmul_%s_t_swiglu" % capi.FMT_NAME[fmt], [("u", N), ("u", K)],
                   [dev.paso(T, 0)] + [dev.matrix(fmt, r, N, K) for r in raw] + [dev.buf(x), y], (1, 1, (T + 31) // 32))
    got = dev.get(y, (T + 1, N))
    assert np.all(got[T] == 7.0)
    g, u = (x.astype(np.float64) @ w.T for w in W)
    silu = g / (1 + np.exp(-g))
    bg, bu = (split_bound(w, x) for w in W)
    assert np.all(np.abs(got[:T] - silu * u) <= 1.1 * bg * (np.abs(u) + bu) + np.abs(silu) * bu + 2.0 ** -20 * np.abs(silu * u))


@pytest.mark.parametrize("op,fmt", [("t", capi.F32), ("4", capi.F32), ("t", capi.Q4_K), ("swiglu", capi.Q4_K)])
def test_operands_past_4_gib(quipu, dev, oracle, op, fmt):
    """62720 token rows of K = 15360 (their operands would take 4.5 GB, past the kernels' offsets): every row like any other.
    All rows are ones but for some at the edges of the passes that such a call is made in and of 4 GiB."""
    T, N, K = 62720, 16, 15360
    rows = np.array([0, 1, 30847, 30848, 30849, 61695, 61696, 62143, 62144, T - 1])
    rng = np.random.default_rng(88)
    xs = (rng.standard_normal((len(rows), K)) / np.sqrt(K)).astype(np.float32)
    raw = [raw_matrix(fmt, N, K, 89 + i) for i in range(2)]
    hw = [dev.matrix(fmt, r, N, K) for r in raw]
    x, y = quipu.alloc(4 * T * K), dev.buf(np.full((T + 1, N), 7.0, np.float32))
    dev.hs.append(x)
    quipu.dispatch("fill_u32", [("u", 0x38000000), ("u", T * K), ("u", 0)], [0, x])  # 2^-15
    for r, v in zip(rows, xs):
        quipu.upload(x, v, int(r) * 4 * K)
    p = dev.paso(T, 0)
    name = "matmul_%s_t_swiglu" % capi.FMT_NAME[fmt] if op == "swiglu" else "matmul_%s_%s" % (capi.FMT_NAME[fmt], op)
    grid = capi.dim2((N + 7) // 8) + ((T + 3) // 4,) if op == "4" else ((N + 63) // 64, 1, (T + 31) // 32)
    quipu.dispatch(name, [("u", N), ("u", K), ("u", 0), ("u", 0)], [p] + hw[:2 if op == "swiglu" else 1] + [x, y], grid)
    got = dev.get(y, (T + 1, N))
    assert np.all(got[T] == 7.0)
    other = np.ones(T, bool)
    other[rows] = False
    assert np.all(got[:T][other] == got[2])
    x64 = np.vstack([xs, np.full((1, K), 2.0 ** -15, np.float32)])
    got = np.vstack([got[rows], got[2:3]])
    W = [weights(oracle, fmt, r, N, K) for r in raw]
    g, u = (x64.astype(np.float64) @ w.T for w in W)
    bg, bu = ((bound if fmt == capi.F32 else split_bound)(w, x64) for w in W)
    if op != "swiglu":
        assert np.all(np.abs(got - g) <= bg)
        return
    silu = g / (1 + np.exp(-np.clip(g, -700, None)))
    assert np.all(np.abs(got - silu * u) <= 1.1 * bg * (np.abs(u) + bu) + np.abs(silu) * bu + 2.0 ** -20 * np.abs(silu * u))


def test_more_than_a_million_rows(quipu, dev):
    """1050000 token rows: more 16-row tiles than a launch's grid takes in one dimension."""
    T, N, K = 1050000, 4, 16
    rng = np.random.default_rng(92)
    raw = raw_matrix(capi.F32, N, K, 93)
    x = rng.standard_normal((T, K), dtype=np.float32)
    W = raw.view(np.float32).reshape(N, K).astype(np.float64)
    assert np.all(np.abs(matmul(quipu, dev, capi.F32, raw, N, K, x) - x.astype(np.float64) @ W.T) <= bound(W, x))


@pytest.mark.parametrize("fmt", KQ)
def test_many_jobs_per_expert(quipu, dev, oracle, fmt):
    """matmul_<fmt>_eg in tiles of 128 jobs: more than 64 experts (their counts are scanned 64 at a time), some without jobs,
    one with every token, others with a few or just over 128; the same bits with and without P[4]."""
    E, N, K, k, T = 70, 130, 512, 3, 700
    rng = np.random.default_rng(86)
    sel = np.stack([np.concatenate([[66], rng.permutation(8)[:2] * 9]) for _ in range(T)]).astype(np.uint32).ravel()
    raw = raw_matrix(fmt, E * N, K, 87)
    W = weights(oracle, fmt, raw, E * N, K).reshape(E, N, K)
    hw = dev.matrix(fmt, raw, E * N, K)
    sb, lb, ob = dev.buf(sel), dev.zeros(4 * T * k), dev.zeros(4 * (E + 1))
    p = dev.paso(T, 0)
    quipu.dispatch("moe_group", [("u", E), ("u", k)], [p, sb, lb, ob])
    for tfijo, m in ((k, 1), (1, k)):
        x = rng.standard_normal((T * k // tfijo, K)).astype(np.float32)
        xb, outs = dev.buf(x), []
        for extra in ([("u", m), ("u", 0)], []):
            y = dev.zeros(4 * T * k * N)
            quipu.dispatch("matmul_%s_eg" % capi.FMT_NAME[fmt], [("u", N), ("u", K), ("u", 0), ("u", tfijo)] + extra,
                           [p, hw, xb, y, lb, ob], ((N + 63) // 64, E, (T + 31) // 32))
            outs.append(dev.get(y, (T * k, N)))
        assert np.array_equal(outs[0], outs[1])
        for e in np.unique(sel):
            js = np.flatnonzero(sel == e)
            xe = x[js // tfijo]
            assert np.all(np.abs(outs[0][js] - xe.astype(np.float64) @ W[e].T) <= bound(W[e], xe)), e


@pytest.mark.parametrize("fmt,T", [(capi.Q4_K, 5), (capi.Q4_K, 100), (capi.Q8_0, 5), (capi.F32, 5)])
@pytest.mark.parametrize("m", [0, 1])
def test_grouped_matmul_in_large_buffers(quipu, dev, oracle, fmt, T, m):
    """matmul_<fmt>_eg on the first rows of buffers with room for 3.7 million (whose operands would take 4 GiB and 2 KB): the
    listed jobs' results, and no workspace that follows the room."""
    import ctypes
    E, N, K, k = 3, 20, 256, 2

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    rng = np.random.default_rng(90)
    sel = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32).ravel()
    raw = raw_matrix(fmt, E * N, K, 91)
    W = weights(oracle, fmt, raw, E * N, K).reshape(E, N, K)
    hw = dev.matrix(fmt, raw, E * N, K)
    wb = [hw, capi.scale_plane(fmt, hw, E * N, K)] if fmt in PLANAR else [hw]
    rows = 233017 * 16
    x, y, lb = quipu.alloc(4 * rows * K), quipu.alloc(4 * rows * k * N), quipu.alloc(4 * 60000)
    dev.hs += [x, y, lb]
    sb, ob, p = dev.buf(sel), dev.zeros(4 * (E + 1)), dev.paso(T, 0)
    xs = rng.standard_normal((T, K)).astype(np.float32)
    quipu.upload(x, xs)
    quipu.dispatch("moe_group", [("u", E), ("u", k)], [p, sb, lb, ob])
    quipu.sync()
    before = free_bytes()
    quipu.dispatch("matmul_%s_eg" % capi.FMT_NAME[fmt], [("u", N), ("u", K), ("u", 0), ("u", k)] + [("u", m)] * (m > 0),
                   [p] + wb + [x, y, lb, ob], ((N + 63) // 64, E, (T + 31) // 32))
    got = dev.get(y, (T * k, N))
    assert before - free_bytes() < 1 << 28
    for j in range(T * k):
        xr = xs[j // k][None]
        assert np.all(np.abs(got[j] - (xr.astype(np.float64) @ W[sel[j]].T)[0]) <= split_bound(W[sel[j]], xr)[0]), j


def test_grouped_matmul_of_a_list_in_a_large_buffer(quipu, dev, oracle):
    """A job list at the start of a 2 GiB buffer: the launch follows the jobs that the dispatch can have, not the room (20
    million empty tiles took 5 ms; the call itself is below 0.1 ms)."""
    import ctypes
    fmt, E, N, K, k, T = capi.Q4_K, 3, 600, 256, 2, 100
    rng = np.random.default_rng(94)
    sel = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32).ravel()
    raw = raw_matrix(fmt, E * N, K, 95)
    W = weights(oracle, fmt, raw, E * N, K).reshape(E, N, K)
    jobs = [np.flatnonzero(sel == e) for e in range(E)]
    off = np.cumsum([0] + [len(j) for j in jobs]).astype(np.uint32)
    lst = quipu.alloc(2 << 30)
    dev.hs.append(lst)
    quipu.upload(lst, np.concatenate(jobs).astype(np.uint32))
    x = rng.standard_normal((T, K)).astype(np.float32)
    y = dev.zeros(4 * T * k * N)
    b = [dev.paso(T, 0), dev.matrix(fmt, raw, E * N, K), dev.buf(x), y, lst, dev.buf(off)]
    ev = [ctypes.c_uint64(), ctypes.c_uint64()]
    for e in ev:
        quipu.L.qp_event_create(ctypes.byref(e))
    best = 1e9
    for _ in range(3):
        quipu.L.qp_event_record(ev[0])
        quipu.dispatch("matmul_q4k_eg", [("u", N), ("u", K), ("u", 0), ("u", k), ("u", 1)], b, ((N + 63) // 64, E, (T + 31) // 32))
        quipu.L.qp_event_record(ev[1])
        ms = ctypes.c_float()
        quipu.L.qp_event_elapsed(ev[0], ev[1], ctypes.byref(ms))
        best = min(best, ms.value)
    for e in ev:
        quipu.L.qp_event_free(e)
    got = dev.get(y, (T * k, N))
    for j in range(T * k):
        assert np.all(np.abs(got[j] - W[sel[j]] @ x[j // k].astype(np.float64)) <= bound(W[sel[j]], x[j // k][None])[0]), j
    assert best < 2.0, best


@pytest.mark.parametrize("f16", [0, 1])
@pytest.mark.parametrize("hd,nh,nkv,T,pos0,swa,cap", [
    (128, 8, 8, 1, 0, 0, 0),          # one key
    (64, 6, 2, 5, 31, 0, 0),          # a group of 3 heads, 15 rows, keys to a tile's edge
    (128, 8, 4, 8, 1000, 0, 0),       # 16 rows, keys shared out
    (128, 10, 2, 7, 64, 0, 0),        # 35 rows: the second block of 32 nearly empty
    (64, 32, 1, 3, 500, 0, 0),        # 32 heads per KV head
    (128, 4, 2, 70, 130, 33, 0),      # a window narrower than a block, no ring
    (64, 8, 2, 24, 200, 64, 88),      # a ring of 88 slots (no multiple of 32) that the keys wrap in
    (128, 4, 4, 1, 500, 100, 132),    # one token of a ring
    (64, 4, 4, 40, 0, 64, 104),       # a ring that is not full yet
])
def test_attention_any_cache(quipu, dev, hd, nh, nkv, T, pos0, swa, cap, f16):
    """atencion on f32 caches, windows and rings against float64: keys a row does not see (later ones, those before its
    window, ring slots not written) are NaN or 6e4 in the cache and must not matter.

    Bound: scores are exact to 2^-21 |q| |k| scale (22-bit factors, products and sums in float32), so weights to that
    relative error e; outputs to (2 e + 2^-19) max |v| (22-bit probabilities and values, float32 sums over the keys)."""
    kvd, n = nkv * hd, pos0 + T
    rng = np.random.default_rng(81)
    q = rng.standard_normal((T, nh * hd)).astype(np.float32)
    kf, vf = (rng.standard_normal((n, kvd)).astype(np.float32) * 10.0 ** rng.uniform(-2, 1, (n, 1)).astype(np.float32)
              for _ in range(2))
    dt = np.float16 if f16 else np.float32
    kf, vf = kf.astype(dt).astype(np.float32), vf.astype(dt).astype(np.float32)
    slots = cap or n + 9
    # (the f16 path without windows takes slots not yet written as finite: the engine zeroes its caches)
    kc, vc = (np.full((slots, kvd), 0 if f16 and not swa and nh // nkv in (1, 2, 4, 8) else np.nan, dt) for _ in range(2))
    for p in range(max(0, n - slots), n):
        kc[p % slots], vc[p % slots] = kf[p], vf[p]
    if swa and not cap:
        kc[:max(0, pos0 + 1 - swa)] = 6e4  # before every row's window
    if f16:
        import refs
        vb = dev.buf(refs.v_tiled(vc, kvd))
    else:
        vb = dev.buf(vc)
    o = dev.zeros(4 * T * nh * hd)
    scale = float(np.float32(1 / np.sqrt(hd)))
    quipu.dispatch("atencion", [("u", hd), ("u", nh), ("u", nkv), ("u", swa), ("f", scale), ("u", cap), ("u", 0), ("u", 0),
                                ("u", f16), ("u", slots)],
                   [dev.paso(T, pos0), dev.buf(q), dev.buf(kc), vb, o], (nh, T))
    got = dev.get(o, (T, nh, hd))
    q64, k64, v64 = (a.astype(np.float64).reshape(a.shape[0], -1, hd) for a in (q, kf, vf))
    for t in range(T):
        a, b = max(0, pos0 + t + 1 - swa) if swa else 0, pos0 + t + 1
        for h in range(nh):
            k, v = k64[a:b, h * nkv // nh], v64[a:b, h * nkv // nh]
            s = k @ q64[t, h] * scale
            w = np.exp(s - s.max())
            w /= w.sum()
            e = 2.0 ** -21 * np.abs(q64[t, h]).max() * np.abs(k).max() * hd * scale
            assert np.all(np.abs(got[t, h] - w @ v) <= (2 * e + 2.0 ** -19) * np.abs(v).max()), (t, h)


@pytest.mark.parametrize("f16", [0, 1])
@pytest.mark.parametrize("hd,nh,nkv,T,pos0,swa,cap", [(128, 8, 4, 24, 40, 0, 0),   # two blocks of 32 rows, f32 or window
                                                      (64, 4, 4, 9, 300, 40, 64),   # a block of 16 rows, a ring
                                                      (128, 6, 2, 1, 700, 600, 0)])  # one token, keys shared out
@pytest.mark.parametrize("kind", ["k_infinite", "k_minus_infinite", "k_huge", "v_huge", "v_without_weight", "q_spread", "blocks"])
def test_attention_unlike_magnitudes(quipu, dev, hd, nh, nkv, T, pos0, swa, cap, f16, kind):
    """Keys and values far larger than the others, infinities among them: a row that does not see such a key, or gives it
    no weight, has the result that it would have without it.

    Bound as in test_attention_any_cache, over the keys with a weight above 1e-36 only (below it a weight is 0 in float32)."""
    if f16 and not swa:
        swa = 1000  # (f16 caches without a window take another kernel)
    rng = np.random.default_rng(83)
    kvd, n = nkv * hd, pos0 + T
    q = rng.standard_normal((T, nh, hd)).astype(np.float32)
    q[..., 0] = 4.0
    kf, vf = (rng.standard_normal((n, kvd)).astype(np.float32) for _ in range(2))
    late = pos0 + T // 2  # seen by the later half of the chunk only (one token: by that token)
    big = np.float32(6e4 if f16 else 2.0 ** 60)
    if kind == "k_infinite":
        kf[late, 5::hd] = np.inf
    elif kind == "k_minus_infinite":
        kf[late, 0::hd] = -np.inf  # (q's first input is positive: no weight)
    elif kind == "k_huge":
        kf[late, 7::hd] = big
    elif kind == "v_huge":
        vf *= np.float32(1e-3)
        vf[late] = big
    elif kind == "v_without_weight":
        vf *= np.float32(1e-3)
        vf[pos0 - 3] = big
        kf[pos0 - 3] = 0
        kf[pos0 - 3, 0::hd] = -3000
    elif kind == "blocks":  # magnitudes that change forth and back along the keys
        kf[::37] *= np.float32(1e-6)
        vf[n // 2:n // 2 + 200] *= np.float32(1e-4 if f16 else 1e-7)
    else:
        q[T // 2:, :, 3] *= np.float32(2.0 ** 30)
        kf[:, 3::hd] = 0
    dt = np.float16 if f16 else np.float32
    kf, vf = kf.astype(dt).astype(np.float32), vf.astype(dt).astype(np.float32)
    slots = cap or n + 9
    kc, vc = (np.full((slots, kvd), np.nan, dt) for _ in range(2))
    for p in range(max(0, n - slots), n):
        kc[p % slots], vc[p % slots] = kf[p], vf[p]
    import refs
    o = dev.zeros(4 * T * nh * hd)
    scale = float(np.float32(1 / np.sqrt(hd)))
    quipu.dispatch("atencion", [("u", hd), ("u", nh), ("u", nkv), ("u", swa), ("f", scale), ("u", cap), ("u", 0), ("u", 0),
                                ("u", f16), ("u", slots)],
                   [dev.paso(T, pos0), dev.buf(q), dev.buf(kc), dev.buf(refs.v_tiled(vc, kvd) if f16 else vc), o], (nh, T))
    got = dev.get(o, (T, nh, hd))
    q64, k64, v64 = q.astype(np.float64), *(a.astype(np.float64).reshape(n, nkv, hd) for a in (kf, vf))
    for t in range(T):
        a, b = max(0, pos0 + t + 1 - swa) if swa else 0, pos0 + t + 1
        for h in range(nh):
            k, v = k64[a:b, h * nkv // nh], v64[a:b, h * nkv // nh]
            s = k @ q64[t, h] * scale
            if s.max() == np.inf:
                assert not np.isfinite(got[t, h]).any(), (t, h)
                continue
            w = np.exp(s - s.max())
            w /= w.sum()
            on = w > 1e-36
            e = 2.0 ** -21 * (np.abs(k[on]) @ np.abs(q64[t, h])).max() * scale
            assert np.all(np.abs(got[t, h] - w[on] @ v[on]) <= (2 * e + 2.0 ** -19) * np.abs(v[on]).max()), (t, h)


def test_attention_shares_cover_no_token_past_the_dispatch(quipu, dev):
    """A Paso of more tokens than the dispatch covers: the others' outputs stay as they were (shares of the keys keep
    partial states for the covered tokens only)."""
    hd, nh, nkv, rows = 64, 2, 1, 600
    rng = np.random.default_rng(82)
    q, kc, vc = (rng.standard_normal(s).astype(np.float32) for s in ((9, nh * hd), (rows, hd), (rows, hd)))
    o = dev.buf(np.full((9, nh * hd), 5.0, np.float32))
    quipu.dispatch("atencion", [("u", hd), ("u", nh), ("u", nkv), ("u", 0), ("f", 0.125), ("u", 0), ("u", 0), ("u", 0),
                                ("u", 0), ("u", rows)],
                   [dev.paso(9, 500), dev.buf(q), dev.buf(kc), dev.buf(vc), o], (nh, 2))
    got = dev.get(o, (9, nh * hd))
    assert np.all(got[2:] == 5.0) and not np.any(got[:2] == 5.0)


@pytest.mark.parametrize("V,k", [(5, 4), (2047, 128), (2050, 100), (6145, 40), (128256, 128)])
@pytest.mark.parametrize("kind", ["equal", "few", "infinite", "signs", "nan"])
def test_topk_equal_values(quipu, dev, V, k, kind):
    """topk_cand where values repeat within a chunk of 2048, across chunks and at the limit: the lower ids first, +0 before
    -0, infinities at their ends, and the flags (bit 1: equal values among the k + 1 largest, bit 0: a NaN)."""
    rng = np.random.default_rng(V + k)
    v = {"equal": np.full(V, -3.25), "few": rng.integers(-2, 3, V) * 0.5, "infinite": np.where(rng.random(V) < 0.5, -np.inf, 1.0),
         "signs": np.where(rng.random(V) < 0.5, -0.0, 0.0), "nan": np.zeros(V)}[kind].astype(np.float32)
    if kind == "infinite":
        v[V // 2] = np.inf
    if kind == "nan":
        v.view(np.uint32)[:] = 0xffffffff
        assert topk_cand(quipu, dev, v, k)[0] & 1
        return
    flags, kk, vals, ids = topk_cand(quipu, dev, v, k)
    order = np.lexsort((np.arange(V), np.signbit(v), -v))[:k + 1]
    assert kk == k and flags == (2 if (v[order[:-1]] == v[order[1:]]).any() else 0)
    assert ids.tolist() == order[:k].tolist()
    assert vals.view(np.uint32).tolist() == v[order[:k]].view(np.uint32).tolist()


@pytest.mark.parametrize("E,k,T", [(1, 1, 1), (63, 8, 5), (64, 64, 3), (65, 2, 130), (256, 64, 7), (257, 8, 3), (300, 70, 2)])
def test_moe_topk_sizes(quipu, dev, oracle, E, k, T):
    """moe_topk by a wavefront per token (E <= 256, k <= 64) and by a workgroup: the experts exactly, equal logits to the
    lower index; the weights to the exponential's and the sums' rounding (as test_swiglu_moe_ops)."""
    lg = np.random.default_rng(E + k).integers(-12, 13, (T, E)).astype(np.float32) * np.float32(0.5)
    sel, wts = dev.zeros(T * k * 4), dev.zeros(T * k * 4)
    quipu.dispatch("moe_topk", [("u", E), ("u", k), ("u", 1), ("f", 1.5)], [dev.paso(T, 0), dev.buf(lg), sel, wts],
                   ((T + 63) // 64,))
    s_want, w_want = oracle.moe_topk(lg, E, k, 1, 1.5)
    np.testing.assert_array_equal(dev.get(sel, (T * k,), np.uint32), s_want)
    np.testing.assert_allclose(dev.get(wts, (T * k,)), w_want, rtol=2e-6, atol=1e-7)
