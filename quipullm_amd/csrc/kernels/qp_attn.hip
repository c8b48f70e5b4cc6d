// Causal attention over f32 caches, sliding windows and rings (the reference's atencion, gpu.js:467-539) on the matrix
// cores.
//
// A workgroup takes 16 RG (query, head) rows of one KV head and a share of the key tiles of 32 slots, dealt to its four
// wavefronts; each keeps its own softmax state and they meet in LDS.  Scores are S^T = K Q^T and outputs O^T += V^T P^T
// with v_mfma_f32_16x16x32_f16: a lane holds 8 scores of one row, which are its operand of the second product.  Every
// f32 operand is an f16 high and low part (22 bits, two fewer than f32) below a power of two: of the row for Q, 16 times
// the wavefront's first tile's largest magnitude for K and V, 2^10 for P.  Three products per pair (high high, high low,
// low high; low low lies below the sums' rounding); f16 caches need two.  Scores, sums, maxima and outputs are f32,
// probabilities 2^x in f32 before their split.  Distance from 64 bits (2-norm, 128 dimensions, random operands): one token
// behind 3000 keys 3.4e-7, 32 behind 480 3.1e-7, 333 behind 1000 3.3e-7; the general kernel's f32 sums 1.1e-6, 5.6e-7, 7.2e-7.
//
// One scale for several keys is only sound while their magnitudes are alike: a row must not lose bits to a key that it
// does not see, or gives no weight.  So each lane compares its pieces of the operands (32 inputs of a query or key, 4 or 8
// of a value) with that scale: where one lies above it (an infinity always does) or is not zero and below 2^-14 of it, the
// wavefront takes its remaining tiles in f32 (v_mfma_f32_16x16x4_f32 on the same registers, an eighth of the rate or less).
// (A NaN needs no such care: it stays with its key and its row, and in a value it reaches every row of the block either way.)
// The comparisons cost 0 to 1 % of a pass: two windowed layers at 500 tokens 1119 us, 1107 without them.  A first token with
// values 2^16 below the others', whose tile is a quarter of the wavefronts' first: 333 tokens behind 1000 keys 115 us for 95.
// (Returning to the scaled tiles after such a tile: 103, but 101 for ordinary values.)
#include "qp_ints.h"

QP_DEV f32x4 ax_mfma(h8 a, h8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
QP_DEV f32x4 ax_mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// f16 high and low parts of eight values already below 2^10.
QP_DEV void ax_split(const float* v, float up, h8& hi, h8& lo) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float s = v[i] * up;
        hi[i] = (_Float16)s;
        lo[i] = (_Float16)(s - (float)hi[i]);
    }
}
// Exponent e of a magnitude, clamped so that 2^(9 - e) and 2^(e - 9) are normal; -117 for 0.
QP_DEV int ax_exp(float m) {
    const int e = (int)((__float_as_uint(m) >> 23) & 255) - 127;
    return e < -117 ? -117 : e;
}
QP_DEV float ax_pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }
// Magnitudes that operands scaled by 2^(9 - e) may have: below 2^(e + 1), and from 2^(e - 14) on.
QP_DEV float ax_top(int e) { return __uint_as_float((uint32_t)(min(e + 1, 128) + 127) << 23); }
QP_DEV float ax_low(int e) { return __uint_as_float(e - 14 > -127 ? (uint32_t)(e - 14 + 127) << 23 : 1u); }
// The scale of a wavefront's tiles, from the largest magnitude of the first: 16 times it (finite values only).
QP_DEV int ax_anchor(float mx, uint32_t lane) {
    return min(__builtin_amdgcn_readfirstlane(ax_exp(wave_max_v(fminf(mx, 3.4e38f), lane))) + 4, 127);
}

constexpr float AX_LOG2E = 1.4426950408889634f;

typedef uint16_t us2 __attribute__((ext_vector_type(2)));

template <int HD, bool F16, int RG>
QP_DEV void attn_x_body(const QpAttnArgs& a) {
    constexpr int KS = HD / 32, DT = HD / 16;  // steps of 32 dimensions, tiles of 16 (DT dimensions per lane of 16)
    extern __shared__ float4 ax_lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n16 = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t T = min(paso_T(a.paso), a.tcov), pos0 = paso_pos(a.paso);
    const uint32_t G = a.nh / a.nkv, kvh = blockIdx.x, kvd = a.nkv * HD, nrow = T * G;
    const uint32_t r0 = blockIdx.y * (16 * RG);
    if (r0 >= nrow) return;
    const uint32_t t_lo = r0 / G, t_hi = (min(r0 + 16 * RG, nrow) - 1) / G;
    // ---- the rows' queries
    h8 qh[RG][KS], ql[RG][KS];
    float qs[RG];         // score = accumulator * qs (times the keys' scale), in units of log2
    int lim[RG], low[RG]; // keys low < key <= lim
    bool alike = true;    // the operands so far are of like magnitudes (this lane's)
#pragma unroll
    for (int r = 0; r < RG; r++) {
        const uint32_t row = r0 + r * 16 + n16, rc = min(row, nrow - 1), t = rc / G, h = kvh * G + rc % G;
        float v[KS][8];
        float mine = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const uint64_t at = a.q + 4 * (((uint64_t)t * a.nh + h) * HD + s * 32 + g * 8);
            const float4 x = gload<float4>(at), y = gload<float4>(at + 16);
            const float w[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                v[s][i] = w[i];
                mine = fmaxf(mine, fabsf(w[i]));
            }
        }
        float all = fmaxf(mine, bfly_f<4>(mine, lane));
        all = fmaxf(all, bfly_f<5>(all, lane));
        const int e = ax_exp(all);
        alike = alike & (all < __builtin_inff()) & ((mine == 0.0f) | (mine >= ax_low(e)));
#pragma unroll
        for (int s = 0; s < KS; s++) ax_split(v[s], ax_pow2(9 - e), qh[r][s], ql[r][s]);
        qs[r] = ax_pow2(e - 9) * a.scale * AX_LOG2E;
        lim[r] = (int)(pos0 + t);
        low[r] = a.swa && pos0 + t >= a.swa ? (int)(pos0 + t - a.swa) : -1;
    }
    // ---- the key tiles: keys kbeg .. kend in slots first .. (ring: then 0 ..), whole tiles of 32 slots
    const uint32_t kend = a.cap ? pos0 + t_hi + 1 : min(pos0 + t_hi + 1, a.rows);
    const uint32_t kbeg = a.swa && pos0 + t_lo + 1 > a.swa ? min(pos0 + t_lo + 1 - a.swa, kend) : 0;
    const uint32_t first = a.cap ? kbeg % a.cap : kbeg, nkey = a.cap ? min(kend - kbeg, a.cap) : kend - kbeg;
    const uint32_t end_a = a.cap ? min(first + nkey, a.cap) : first + nkey, end_b = first + nkey - end_a;
    const uint32_t ta = nkey ? (end_a + 31) / 32 - first / 32 : 0, nt = ta + (end_b + 31) / 32;
    const uint32_t per = (nt + a.nsplit - 1) / a.nsplit, i0 = blockIdx.z * per, i1 = min(nt, i0 + per);
    constexpr uint32_t eb = F16 ? 2 : 4;
    const uint64_t slots = F16 ? (a.rows + 31ull) / 32 * 32 : a.rows;  // (the f16 value cache holds whole tiles)
    const __amdgpu_buffer_rsrc_t kr = kq_rsrc(a.kc, (uint64_t)a.rows * kvd * eb), vr = kq_rsrc(a.vc, slots * kvd * eb);

    constexpr int KL = F16 ? KS : 2 * KS;       // 16-byte loads of one key per lane
    constexpr int VL = F16 ? DT : 8 * (DT / 4); // 16-byte loads of a tile's values per lane
    u32x4 kw[2][KL], vw[VL];
    struct Tile { uint32_t slot, lo, hi; int off; };  // slots lo .. hi of it hold keys slot + off
    auto tile = [&](uint32_t i) __attribute__((always_inline)) {
        Tile t;
        if (i < ta) t = {(first / 32 + i) * 32, first, end_a, (int)(kbeg - first)};
        else t = {(i - ta) * 32, 0, end_b, (int)(kbeg + a.cap - first)};
        return t;
    };
    auto load_k = [&](uint32_t i) __attribute__((always_inline)) {
        const Tile t = tile(i);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t s = t.slot + h * 16 + n16;
            const uint32_t o = i < i1 && s >= t.lo && s < t.hi ? (s * kvd + kvh * HD + 8 * g) * eb : QP_NOOFF;
#pragma unroll
            for (int c = 0; c < KL; c++)
                kw[h][c] = __builtin_amdgcn_raw_buffer_load_b128(kr, o, F16 ? c * 64 : (c >> 1) * 128 + (c & 1) * 16, 0);
        }
    };
    auto load_v = [&](uint32_t i) __attribute__((always_inline)) {
        const Tile t = tile(i);
        if constexpr (F16) {
            const uint32_t o = i < i1 ? (t.slot * kvd + (kvh * HD + DT * n16) * 32) * 2 + g * 16 : QP_NOOFF;
#pragma unroll
            for (int c = 0; c < DT; c++) vw[c] = __builtin_amdgcn_raw_buffer_load_b128(vr, o, c * 64, 0);
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t s = t.slot + (j >> 2) * 16 + 4 * g + (j & 3);
                const uint32_t o = i < i1 && s >= t.lo && s < t.hi ? (s * kvd + kvh * HD + DT * n16) * 4 : QP_NOOFF;
#pragma unroll
                for (int c = 0; c < DT / 4; c++)
                    vw[j * (DT / 4) + c] = __builtin_amdgcn_raw_buffer_load_b128(vr, o, c * 16, 0);
            }
        }
    };

    // value x (of 8) of step c of the lane's key h, and the lane's key j's value at dimension d
    auto key = [&](int h, int c, int x) __attribute__((always_inline)) -> float {
        if constexpr (F16) return h2f(kw[h][c][x >> 1] >> (16 * (x & 1)));
        else return __uint_as_float(kw[h][2 * c + (x >> 2)][x & 3]);
    };
    auto val = [&](int j, int d) __attribute__((always_inline)) -> float {
        if constexpr (F16) return h2f(vw[d][j >> 1] >> (16 * (j & 1)));
        else return __uint_as_float(vw[j * (DT / 4) + (d >> 2)][d & 3]);
    };
    // the f16 caches' largest magnitudes, two halves at a time
    auto pk_max = [&](uint32_t m, uint32_t w) __attribute__((always_inline)) -> uint32_t {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2, m), __builtin_bit_cast(us2, w & 0x7fff7fffu)));
    };

    f32x4 o[RG][DT];
    float m[RG], l[RG], p[RG][8], corr[RG];
    int ek = 0, ev = 0;     // the keys' and values' scale
#pragma unroll
    for (int r = 0; r < RG; r++) {
        m[r] = -3.0e38f;
        l[r] = 0.0f;
#pragma unroll
        for (int d = 0; d < DT; d++) o[r][d] = f32x4{0, 0, 0, 0};
    }
    // softmax of the lane's 8 keys of each of its rows: scores s times unit (and qs), in units of log2
    auto softmax = [&](const Tile& t, const f32x4 (&s)[RG][2], auto Split, float unit) __attribute__((always_inline)) {
        // all slots hold keys that every row of the block sees
        const bool whole = t.slot >= t.lo && t.slot + 32 <= t.hi && (int)t.slot + 31 + t.off <= (int)(pos0 + t_lo) &&
                           (!a.swa || (int)t.slot + t.off > (int)(pos0 + t_hi) - (int)a.swa);
#pragma unroll
        for (int r = 0; r < RG; r++) {
            const float c = Split.v ? qs[r] * unit : unit;
            float x[8], mx = -3.0e38f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                x[j] = s[r][j >> 2][j & 3] * c;
                if (!whole) {
                    const uint32_t sl = t.slot + (j >> 2) * 16 + 4 * g + (j & 3);
                    const int key = (int)sl + t.off;
                    x[j] = sl >= t.lo && sl < t.hi && key <= lim[r] && key > low[r] ? x[j] : -__builtin_inff();
                }
                mx = fmaxf(mx, x[j]);
            }
            mx = fmaxf(mx, bfly_f<4>(mx, lane));
            mx = fmaxf(mx, bfly_f<5>(mx, lane));
            const float mn = fmaxf(m[r], mx);
            corr[r] = __builtin_amdgcn_exp2f(m[r] - mn);
            m[r] = mn;
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                p[r][j] = __builtin_amdgcn_exp2f(x[j] - mn);
                sum += p[r][j];
            }
            l[r] = l[r] * corr[r] + sum;
        }
    };
    // f16 values: slots without a key may hold anything
    auto mask_v = [&](const Tile& t) __attribute__((always_inline)) {
        if (!F16 || (t.slot >= t.lo && t.slot + 32 <= t.hi)) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t sl = t.slot + (j >> 1) * 16 + 4 * g + 2 * (j & 1);
            const uint32_t keep = (sl >= t.lo && sl < t.hi ? 0xffffu : 0u) | (sl + 1 >= t.lo && sl + 1 < t.hi ? 0xffff0000u : 0u);
#pragma unroll
            for (int d = 0; d < VL; d++) vw[d][j] &= keep;
        }
    };
    auto rescale = [&](float f) __attribute__((always_inline)) {
        bool same = f == 1.0f;
#pragma unroll
        for (int r = 0; r < RG; r++) same = same && corr[r] == 1.0f;
        if (__all(same)) return;
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int x = 0; x < 4; x++) o[r][d][x] *= corr[r] * f;
    };
    auto pv_f32 = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int r = 0; r < RG; r++) o[r][d] = ax_mfma(val(j, d), p[r][j], o[r][d]);
    };
    uint32_t i = i0 + wave;
    load_k(i);
    load_v(i);
    bool first_tile = true, pending = false;  // pending: tile i's scores are done, its values not
    for (; i < i1; i += 4) {
        const Tile t = tile(i);
        // ---- S^T = K Q^T
        if constexpr (F16) {  // (a key's rounding is its own: only infinities matter)
            uint32_t mx = 0;
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int c = 0; c < KL; c++)
#pragma unroll
                    for (int x = 0; x < 4; x++) mx = pk_max(mx, kw[h][c][x]);
            alike = alike & ((mx & 0xffffu) < 0x7c00u) & ((mx >> 16) < 0x7c00u);
        } else {
            float kx[2] = {0.0f, 0.0f};
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int c = 0; c < KS; c++)
#pragma unroll
                    for (int x = 0; x < 8; x++) kx[h] = fmaxf(kx[h], fabsf(key(h, c, x)));
            if (first_tile) ek = ax_anchor(fmaxf(kx[0], kx[1]), lane);
            const float top = ax_top(ek), lo = ax_low(ek);
#pragma unroll
            for (int h = 0; h < 2; h++) alike = alike & (kx[h] < top) & ((kx[h] == 0.0f) | (kx[h] >= lo));
        }
        if (!__all(alike)) break;
        f32x4 s[RG][2];
        const float upk = F16 ? 1.0f : ax_pow2(9 - ek);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int c = 0; c < KS; c++) {
                h8 kh, kl;
                if constexpr (F16) {
                    kh = __builtin_bit_cast(h8, kw[h][c]);
                } else {
                    float v[8];
#pragma unroll
                    for (int x = 0; x < 8; x++) v[x] = key(h, c, x);
                    ax_split(v, upk, kh, kl);
                }
#pragma unroll
                for (int r = 0; r < RG; r++) s[r][h] = ax_mfma(kh, qh[r][c], c ? s[r][h] : f32x4{0, 0, 0, 0});
#pragma unroll
                for (int r = 0; r < RG; r++) s[r][h] = ax_mfma(kh, ql[r][c], s[r][h]);
                if constexpr (!F16) {
#pragma unroll
                    for (int r = 0; r < RG; r++) s[r][h] = ax_mfma(kl, qh[r][c], s[r][h]);
                }
            }
        load_k(i + 4);
        softmax(t, s, SkInt<1>(), F16 ? 1.0f : ax_pow2(ek - 9));
        // ---- O^T += V^T P^T
        mask_v(t);
        float vx[8];
        if constexpr (F16) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint32_t w = 0;
#pragma unroll
                for (int d = 0; d < DT; d++) w = pk_max(w, vw[d][j]);
                vx[2 * j] = h2f(w);
                vx[2 * j + 1] = h2f(w >> 16);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                vx[j] = 0.0f;
#pragma unroll
                for (int d = 0; d < DT; d++) vx[j] = fmaxf(vx[j], fabsf(val(j, d)));
            }
        }
        if (first_tile) {
            float all = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) all = fmaxf(all, vx[j]);
            ev = ax_anchor(all, lane);
        }
        first_tile = false;
        const float top = ax_top(ev), lo = ax_low(ev);
#pragma unroll
        for (int j = 0; j < 8; j++) alike = alike & (vx[j] < top) & ((vx[j] == 0.0f) | (vx[j] >= lo));
        if (!__all(alike)) {
            pending = true;
            break;
        }
        rescale(1.0f);
        const float upv = F16 ? 1.0f : ax_pow2(9 - ev);
        h8 ph[RG], pl[RG];
#pragma unroll
        for (int r = 0; r < RG; r++) ax_split(p[r], 1024.0f, ph[r], pl[r]);
#pragma unroll
        for (int d = 0; d < DT; d++) {
            h8 vh, vl;
            if constexpr (F16) {
                vh = __builtin_bit_cast(h8, vw[d]);
            } else {
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = val(j, d);
                ax_split(v, upv, vh, vl);
            }
#pragma unroll
            for (int r = 0; r < RG; r++) o[r][d] = ax_mfma(vh, ph[r], o[r][d]);
#pragma unroll
            for (int r = 0; r < RG; r++) o[r][d] = ax_mfma(vh, pl[r], o[r][d]);
            if constexpr (!F16) {
#pragma unroll
                for (int r = 0; r < RG; r++) o[r][d] = ax_mfma(vl, ph[r], o[r][d]);
            }
        }
        load_v(i + 4);
    }
    float back = (F16 ? 1.0f : ax_pow2(ev - 9)) * 0x1p-10f;  // o times it: the outputs
    if (i < i1) {  // the other tiles in f32
        if (!pending) {
#pragma unroll
            for (int r = 0; r < RG; r++) corr[r] = 1.0f;
        }
        rescale(back);
        back = 1.0f;
        if (pending) {
            pv_f32();
            load_v(i + 4);
            i += 4;
        }
        for (; i < i1; i += 4) {
            const Tile t = tile(i);
            f32x4 s[RG][2];
#pragma unroll
            for (int r = 0; r < RG; r++) {
                const uint32_t rc = min(r0 + r * 16 + n16, nrow - 1);
                const uint64_t at = a.q + 4 * (((uint64_t)(rc / G) * a.nh + kvh * G + rc % G) * HD + g * 8);
                s[r][0] = s[r][1] = f32x4{0, 0, 0, 0};
#pragma unroll
                for (int c = 0; c < KS; c++) {
                    const float4 q0 = gload<float4>(at + c * 128), q1 = gload<float4>(at + c * 128 + 16);
                    const float q[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
                    for (int x = 0; x < 8; x++)
#pragma unroll
                        for (int h = 0; h < 2; h++) s[r][h] = ax_mfma(key(h, c, x), q[x], s[r][h]);
                }
            }
            load_k(i + 4);
            softmax(t, s, SkInt<0>(), a.scale * AX_LOG2E);
            mask_v(t);
            rescale(1.0f);
            pv_f32();
            load_v(i + 4);
        }
    }
    // ---- the four wavefronts' states meet: [wave][row][HD + 4], then [wave][row] (m, l)
    constexpr int LD = HD + 4;
    float* ol = reinterpret_cast<float*>(ax_lds);
    float* ml = ol + 4 * RG * 16 * LD;
#pragma unroll
    for (int r = 0; r < RG; r++) {
        float lt = l[r];
        lt += bfly_f<4>(lt, lane);
        lt += bfly_f<5>(lt, lane);
        const uint32_t at = wave * RG * 16 + r * 16 + n16;
        if (g == 0) {
            ml[2 * at] = m[r];
            ml[2 * at + 1] = lt;
        }
        // dimensions DT * (4 g + x) + d of the row
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
            for (int d = 0; d < DT; d += 4)
                *reinterpret_cast<float4*>(ol + at * LD + DT * (4 * g + x) + d) =
                    make_float4(o[r][d][x] * back, o[r][d + 1][x] * back, o[r][d + 2][x] * back, o[r][d + 3][x] * back);
    }
    __syncthreads();
    for (uint32_t k = tid; k < RG * 16 * (HD / 4); k += 256) {
        const uint32_t lr = k / (HD / 4), c = k % (HD / 4), row = r0 + lr;
        if (row >= nrow) continue;
        float M = -3.0e38f;
#pragma unroll
        for (int w = 0; w < 4; w++) M = fmaxf(M, ml[2 * (w * RG * 16 + lr)]);
        float L = 0.0f;
        float4 s = make_float4(0, 0, 0, 0);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t at = w * RG * 16 + lr;
            const float lw = ml[2 * at + 1], f = lw != 0.0f ? __builtin_amdgcn_exp2f(ml[2 * at] - M) : 0.0f;
            const float4 v = *reinterpret_cast<const float4*>(ol + at * LD + 4 * c);
            L += lw * f;
            if (f != 0.0f) s = make_float4(s.x + v.x * f, s.y + v.y * f, s.z + v.z * f, s.w + v.w * f);
        }
        const uint32_t t = row / G, h = kvh * G + row % G;
        const uint64_t at = (uint64_t)t * a.nh + h;
        if (a.nsplit == 1) {
            gstore<float4>(a.o + 4 * (at * HD + 4 * c), make_float4(s.x / L, s.y / L, s.z / L, s.w / L));
        } else {
            gstore<float4>(a.part_o + 4 * ((at * a.nsplit + blockIdx.z) * HD + 4 * c), s);
            if (c == 0) gstore<float2>(a.part_ml + 8 * (at * a.nsplit + blockIdx.z), make_float2(M, L));
        }
    }
}

#define ATTN_X(HD, NAME, F16)                                                                                         \
    KERNEL __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void qp_attn_x_h##HD##_##NAME##_r1(         \
        QpAttnArgs a) { attn_x_body<HD, F16, 1>(a); }                                                                 \
    KERNEL __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1))) void qp_attn_x_h##HD##_##NAME##_r2(         \
        QpAttnArgs a) { attn_x_body<HD, F16, 2>(a); }
ATTN_X(64, f32, false) ATTN_X(128, f32, false) ATTN_X(64, f16, true) ATTN_X(128, f16, true)

// The shares' partial states of each (query, head) row -> o, in their order: grid rows, hd threads (at most 64 shares).
KERNEL __launch_bounds__(128) void qp_attn_x_comb(QpAttnArgs a) {
    __shared__ float wt[64], den;
    const uint32_t t = blockIdx.x / a.nh, d = threadIdx.x, ns = a.nsplit;
    if (t >= paso_T(a.paso)) return;
    const uint64_t row = blockIdx.x, po = a.part_o + 4 * (row * ns * a.hd + d);
    float v[8];
#pragma unroll
    for (uint32_t s = 0; s < 8; s++) v[s] = s < ns ? gload<float>(po + 4ull * s * a.hd) : 0.0f;
    if (d < 64) {
        const float2 ml = d < ns ? gload<float2>(a.part_ml + 8 * (row * ns + d)) : make_float2(-3.0e38f, 0.0f);
        const float M = wave_max_v(ml.x, d), f = ml.y != 0.0f ? __builtin_amdgcn_exp2f(ml.x - M) : 0.0f;
        wt[d] = f;
        const float L = wave_sum_v(ml.y * f, d);
        if (d == 0) den = L;
    }
    __syncthreads();
    float o = 0.0f;
    for (uint32_t s0 = 0; s0 < ns; s0 += 8) {
#pragma unroll
        for (uint32_t s = 0; s < 8; s++)
            if (s0 + s < ns && wt[s0 + s] != 0.0f) o += v[s] * wt[s0 + s];
#pragma unroll
        for (uint32_t s = 0; s < 8; s++) v[s] = s0 + 8 + s < ns ? gload<float>(po + 4ull * (s0 + 8 + s) * a.hd) : 0.0f;
    }
    gstore<float>(a.o + 4 * (row * a.hd + d), o / den);
}
