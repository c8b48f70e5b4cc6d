// Matrix products of a few to a few hundred token rows with quantized weights (matmul_<fmt>_4 / _t / _eg), on the
// matrix cores with the weights taken as integers.
//
// Y[t][n] (+)= sum_k X[t][k] * W[n][k].  Each weight block is a scale times small integers, so the products run on
// v_mfma_f32_16x16x32_f16 with the integers as f16 (exact) and X as f16 high + low parts of the row scaled by a power
// of two per 256 inputs (22 bits): two matrix instructions per pair, and the block's scale multiplies the f32 sum of a
// whole block.  K-quants with 6-bit (or smaller) sub-block scales take scale * quant as the integer (at most 1953, so
// exact in f16) and one f32 scale per 256 inputs; Q6_K's int8 scale * quant reaches 8064, so its integers are a high
// and a low f16 (three instructions); Q8_0 and IQ4_NL scale the sums of each 32 inputs; f32 rows are scaled by a power
// of two per 32 inputs and split like X (the product of the two low parts is left out).
//
// So X (and f32 weights) have 22 bits below the largest of their 256 (32) inputs, not f32's own: an input 2^11 and more
// below that loses bits against the f32 multiply-adds that ran here before.  What an output is off by is mostly its sums'
// rounding, and the matrix cores add in fewer steps: distance from 64 bits (2-norm, N(0, 1) inputs, 2 / 32 / 63 tokens, in
// parentheses the kernels before: f32 multiply-adds below 64 dispatched tokens, then bf16 parts) f32 128 x 2048 1.6e-7 /
// 1.4e-7 / 1.4e-7 (9e-7 / 8e-7 / 4.5e-6), Q4_K 512 x 4096 3.2e-7 (1.1e-6 / 1.2e-6 / 4.2e-6), Q6_K 3.6e-7 (1.2e-6 / 1.1e-6 /
// 4.3e-6), Q8_0 512 x 1024 1.0e-7 (6e-7 / 6e-7 / 4.0e-6), IQ4_NL 1.0e-7 (5e-7 / 6e-7 / 4.3e-6).
//
// A wavefront takes 16 R weight rows and a slice of K and keeps them in registers, so nothing is staged in LDS: the
// lanes of row n (n = lane % 16) load 16-byte chunks of four consecutive blocks (64 contiguous bytes), and a 4 x 4
// exchange of the four lane groups (v_permlane32_swap, v_permlane16_swap) gives lane group g the g-th dword of every
// chunk, its operand of the instruction: inputs 4g..4g+3 and 16+4g..16+4g+3 of each 32.  X is read as operands made
// once by qp_split_f16 in that order.  The K slices of a workgroup's wavefronts are added through LDS at the end.
#include "qp_ints.h"

// A workgroup per (chunk, tile), each of its four wavefronts 64 inputs of the 16 rows.
KERNEL __launch_bounds__(256) void qp_split_f16(QpSplitArgs a) {
    __shared__ float mxs[4][16];
    __shared__ float sums[16][17];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, m = lane & 15;
    const uint32_t ch = blockIdx.x, nch = gridDim.x;
    uint64_t rows = a.mul ? (uint64_t)paso_T(a.paso) * a.mul : pass_T(a.paso, a.tbase, a.rows);
    if (a.mul && rows > a.cap) rows = a.cap;
    const uint32_t row = blockIdx.y * 16 + m;
    if (blockIdx.y * 16 >= rows) return;
    float4 v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t k = ch * 256 + wave * 64 + j * 16 + 4 * g;
        v[j] = make_float4(0, 0, 0, 0);
        if (row >= rows || k >= a.k) continue;
        if (a.mode == 2) {
            const uint64_t at = a.x + ((uint64_t)((k >> 5) * 4 + ((k >> 3) & 3)) * a.prows + row) * 16 + (k & 7) * 2;
            const uint2 h = gload<uint2>(at), l = gload<uint2>(at + 2ull * a.prows * a.k);
            v[j] = make_float4(__uint_as_float(h.x << 16) + __uint_as_float(l.x << 16),
                               __uint_as_float(h.x & 0xffff0000u) + __uint_as_float(l.x & 0xffff0000u),
                               __uint_as_float(h.y << 16) + __uint_as_float(l.y << 16),
                               __uint_as_float(h.y & 0xffff0000u) + __uint_as_float(l.y & 0xffff0000u));
            continue;
        }
        v[j] = gload<float4>(a.x + 4 * ((uint64_t)row * a.k + k));
        if (a.mode == 1) {
            float* f = &v[j].x;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const __bf16 h = (__bf16)f[i];
                f[i] = (float)h + (float)(__bf16)(f[i] - (float)h);
            }
        }
    }
    float mx = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++)
        mx = fmaxf(fmaxf(fmaxf(mx, fabsf(v[j].x)), fmaxf(fabsf(v[j].y), fabsf(v[j].z))), fabsf(v[j].w));
    mx = fmaxf(mx, bfly_f<4>(mx, lane));
    mx = fmaxf(mx, bfly_f<5>(mx, lane));
    if (g == 0) mxs[wave][m] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(mxs[0][m], mxs[1][m]), fmaxf(mxs[2][m], mxs[3][m]));
    // 2^(9 - e) for the largest magnitude's exponent e: the stored values lie below 2^10
    int e = (int)((__float_as_uint(mx) >> 23) & 255) - 127;
    if (mx == 0.0f) e = 9;
    if (e < -117) e = -117;
    const float up = __uint_as_float((uint32_t)(9 - e + 127) << 23);
    const uint64_t base = a.xs + ((uint64_t)blockIdx.y * nch + ch) * XF_CHUNK + (a.mul ? m * 128 + g * 16 : lane * 16);
    const uint32_t low = a.mul ? XF_LOW : 1024;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const float s[8] = {v[2 * j].x * up, v[2 * j].z * up, v[2 * j].y * up, v[2 * j].w * up,
                            v[2 * j + 1].x * up, v[2 * j + 1].z * up, v[2 * j + 1].y * up, v[2 * j + 1].w * up};
        h8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            hi[i] = (_Float16)s[i];
            const float d = s[i] - (float)hi[i];
            lo[i] = (_Float16)(d == d ? d : 0.0f);  // (an infinite value has no remainder)
        }
        gstore<h8>(base + (wave * 2 + j) * 2048, hi);
        gstore<h8>(base + (wave * 2 + j) * 2048 + low, lo);
        float s0 = (s[0] + s[1]) + (s[2] + s[3]), s1 = (s[4] + s[5]) + (s[6] + s[7]);
        s0 += bfly_f<4>(s0, lane);
        s1 += bfly_f<4>(s1, lane);
        s0 += bfly_f<5>(s0, lane);
        s1 += bfly_f<5>(s1, lane);
        if (g == 0) {
            sums[m][wave * 4 + 2 * j] = s0;
            sums[m][wave * 4 + 2 * j + 1] = s1;
        }
    }
    __syncthreads();
    if (wave == 0) {
        h8 sv;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float s = sums[m][(g & 1) * 8 + i];
            const _Float16 h = (_Float16)s;
            const float d = s - (float)h;
            sv[i] = g < 2 ? h : (_Float16)(d == d ? d : 0.0f);
        }
        gstore<h8>(base + 16384, sv);
    } else if (wave == 1 && g == 0) {
        const uint64_t sc = a.xs + (uint64_t)(a.rows >> 4) * nch * XF_CHUNK;
        gstore<float>(sc + 4 * (((uint64_t)blockIdx.y * nch + ch) * 16 + m),
                      __uint_as_float((uint32_t)(e - 9 + 127) << 23));
    }
}

// ------------------------------------------------------------------ lane-group exchanges
// v: lane group g holds 16 bytes of block g.  Result: element b of lane group g = dword g of block b.
QP_DEV u32x4 sk_transpose(u32x4 v) {
    const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return u32x4{(uint32_t)c[0], (uint32_t)c[1], (uint32_t)d[0], (uint32_t)d[1]};
}
// The dword of lane `from` / 4.
QP_DEV uint32_t sk_from(uint32_t v, uint32_t from) { return (uint32_t)__builtin_amdgcn_ds_bpermute((int)from, (int)v); }

// One block of one row, from the point of view of a lane: its dwords t[chunk] of the data chunks and the whole header.
template <int FMT>
struct SkBlock : SkScales<FMT> {
    uint32_t t[SkK<FMT>::NC];

    // The products of this lane's eight inputs of step j (32 inputs).
    template <int j>
    QP_DEV void step(h8& hi, h8& lo) const {
        using S = SkStep<FMT, j>;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            h2 q[2], l[2];
            sk_quad<FMT, j>(t[S::CHUNK + i], S::HIGH >= 0 ? t[S::HIGH + i] : 0u, this->template scale<j, S::AT>(i), q, l);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                hi[4 * i + k] = q[k >> 1][k & 1];
                if constexpr (FMT == QP_Q6_K) lo[4 * i + k] = l[k >> 1][k & 1];
            }
        }
    }
};

// The X operands of one step for the NT token tiles.
template <int NT>
struct SkX {
    h8 hi[NT], lo[NT];
    QP_DEV void load(__amdgpu_buffer_rsrc_t xr, const uint32_t* xo, uint32_t soff, uint32_t low) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            hi[t] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(xr, xo[t], soff, 0));
            lo[t] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(xr, xo[t], soff + low, 0));
        }
    }
};


// Where a wavefront's weights are: a buffer resource over its rows and the offset of this lane's row.
struct SkRows {
    __amdgpu_buffer_rsrc_t w, d;
    uint32_t off, doff;  // QP_NOOFF: no such row
};

// K-quants: groups of four blocks of 256 inputs, group gi0 + i * gs < gi1.
template <int FMT, int NT, int R, class Sc>
QP_DEV void sk_kq(const SkRows (&rw)[R], uint32_t nb, uint32_t gi0, uint32_t gi1, uint32_t gs, __amdgpu_buffer_rsrc_t xr,
                  const uint32_t* xo, uint32_t low, Sc&& scales, f32x4 (&tot)[R][NT]) {
    using F = SkK<FMT>;
    const uint32_t g = (threadIdx.x & 63) >> 4;
    u32x4 w[R][F::NC];
    uint32_t dd[R];
    auto load = [&](uint32_t gi) __attribute__((always_inline)) {
        const uint32_t blk = 4 * gi + g;
        const bool ok = gi < gi1 && blk < nb;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t o = ok && rw[r].off != QP_NOOFF ? rw[r].off + blk * 16 : QP_NOOFF;
#pragma unroll
            for (int c = 0; c < F::NC; c++)
                w[r][c] = __builtin_amdgcn_raw_buffer_load_b128(rw[r].w, o, c * nb * 16, 0);
            dd[r] = 0;
            if constexpr (FMT == QP_Q6_K)
                dd[r] = __builtin_amdgcn_raw_buffer_load_b16(rw[r].d, ok && rw[r].off != QP_NOOFF ? rw[r].doff + blk * 2 : QP_NOOFF, 0, 0);
            if constexpr (FMT == QP_Q2_K)
                dd[r] = __builtin_amdgcn_raw_buffer_load_b32(rw[r].d, ok && rw[r].off != QP_NOOFF ? rw[r].doff + blk * 4 : QP_NOOFF, 0, 0);
        }
    };
    constexpr int PD = NT == 4 ? 2 : 4;  // steps of X in flight
    SkX<NT> x[PD];
    load(gi0);
#pragma unroll
    for (int j = 0; j < PD; j++) x[j].load(xr, xo, 4 * gi0 * XF_CHUNK + j * 2048, low);
    for (uint32_t gi = gi0; gi < gi1; gi += gs) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < F::NC; c++)
                if (c != F::HDR) w[r][c] = sk_transpose(w[r][c]);
        // (a loop, not four copies: the code of a group that most wavefronts run once would come from memory each time)
        const uint32_t b1 = min(4u, nb - 4 * gi);
#pragma clang loop unroll(disable)
        for (uint32_t b = 0; b < b1; b++) {
            const uint32_t ch = 4 * gi + b, from = (b * 16 + (threadIdx.x & 15)) * 4;
            {
                SkBlock<FMT> blk[R];
#pragma unroll
                for (int r = 0; r < R; r++) {
#pragma unroll
                    for (int c = 0; c < F::NC; c++)
                        if (c != F::HDR) {
                            blk[r].t[c] = w[r][c][0];
                            w[r][c] = u32x4{w[r][c][1], w[r][c][2], w[r][c][3], 0};
                        }
#pragma unroll
                    for (int i = 0; i < 4; i++) blk[r].h[i] = sk_from(w[r][F::HDR][i], from);
                    blk[r].dd = 0;
                    if constexpr (FMT == QP_Q6_K || FMT == QP_Q2_K) blk[r].dd = sk_from(dd[r], from);
                    blk[r].setup();
                }
                const uint32_t so = ch * XF_CHUNK;
                f32x4 p[R][NT];
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int t = 0; t < NT; t++) p[r][t] = f32x4{0, 0, 0, 0};
                // the block after this one (of the next group: its first; none left: this one again)
                const uint32_t nx = b + 1 < b1 ? ch + 1 : gi + gs < gi1 ? 4 * (gi + gs) : ch;
                f32x4 s[NT];
                scales(ch, s);
                h8 xs[NT];
                if constexpr (F::MIN) {
#pragma unroll
                    for (int t = 0; t < NT; t++)
                        xs[t] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(xr, xo[t], so + 16384, 0));
                }
                auto step = [&](auto J) __attribute__((always_inline)) {
                    constexpr int j = decltype(J)::v;
                    SkX<NT>& X = x[j % PD];
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        h8 hi, lo;
                        blk[r].template step<j>(hi, lo);
#pragma unroll
                        for (int t = 0; t < NT; t++) p[r][t] = sk_mfma(X.hi[t], hi, p[r][t]);
#pragma unroll
                        for (int t = 0; t < NT; t++) p[r][t] = sk_mfma(X.lo[t], hi, p[r][t]);
                        if constexpr (F::LO) {
#pragma unroll
                            for (int t = 0; t < NT; t++) p[r][t] = sk_mfma(X.hi[t], lo, p[r][t]);
                        }
                    }
                    X.load(xr, xo, j + PD < 8 ? so + (j + PD) * 2048 : nx * XF_CHUNK + (j + PD - 8) * 2048, low);
                    __builtin_amdgcn_sched_barrier(0xf);  // (the loads stay at their step: hoisted, they would spill)
                };
                step(SkInt<0>()); step(SkInt<1>()); step(SkInt<2>()); step(SkInt<3>());
                step(SkInt<4>()); step(SkInt<5>()); step(SkInt<6>()); step(SkInt<7>());
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const float d = blk[r].d() * (float)(1 << (19 - F::UP));
                    if constexpr (F::MIN) {
                        const h8 mn = blk[r].mins(g);
                        const float dm = blk[r].dmin();
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            const f32x4 mv = sk_mfma(xs[t], mn, f32x4{0, 0, 0, 0});
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                tot[r][t][i] = fmaf(s[t][i], fmaf(d, p[r][t][i], -(dm * mv[i])), tot[r][t][i]);
                        }
                    } else {
#pragma unroll
                        for (int t = 0; t < NT; t++)
#pragma unroll
                            for (int i = 0; i < 4; i++) tot[r][t][i] = fmaf(s[t][i], d * p[r][t][i], tot[r][t][i]);
                    }
                }
            }
        }
        if (gi + gs < gi1) load(gi + gs);
    }
}

// Q8_0, IQ4_NL and f32: chunks of 256 inputs ch0 + i * cs < ch1; the scale of each 32 inputs multiplies their sums.
template <int FMT, int NT, int R, class Sc>
QP_DEV void sk_pl(const SkRows (&rw)[R], uint32_t K, uint32_t ch0, uint32_t ch1, uint32_t cs, __amdgpu_buffer_rsrc_t xr,
                  const uint32_t* xo, uint32_t low, Sc&& scales, f32x4 (&tot)[R][NT]) {
    constexpr int NL = FMT == QP_F32 ? 16 : FMT == QP_Q8_0 ? 4 : 2;  // 16-byte loads per lane and chunk
    const uint32_t g = (threadIdx.x & 63) >> 4;
    const uint32_t rowb = FMT == QP_F32 ? 4 * K : FMT == QP_Q8_0 ? K : K / 2;  // bytes of a row (without scales)
    u32x4 w[R][NL];
    uint32_t dq[R][8];
    auto load = [&](uint32_t ch) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const bool ok = ch < ch1 && rw[r].off != QP_NOOFF;
#pragma unroll
            for (int i = 0; i < NL; i++) {
                const uint32_t in = ch * (256 / 16 * NL * 4) + i * 64 + g * 16;  // byte inside the row
                w[r][i] = __builtin_amdgcn_raw_buffer_load_b128(rw[r].w, ok && in < rowb ? rw[r].off + in : QP_NOOFF, 0, 0);
            }
            if constexpr (FMT != QP_F32) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t blk = ch * 8 + j;
                    dq[r][j] = __builtin_amdgcn_raw_buffer_load_b16(rw[r].d, ok && blk * 32 < K ? rw[r].doff + blk * 2 : QP_NOOFF, 0, 0);
                }
            }
        }
    };
    load(ch0);
    for (uint32_t ch = ch0; ch < ch1; ch += cs) {
        u32x4 c[R][NL];
        float ds[R][8];
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int i = 0; i < NL; i++) c[r][i] = FMT == QP_F32 ? w[r][i] : sk_transpose(w[r][i]);
            if constexpr (FMT != QP_F32) {
#pragma unroll
                for (int j = 0; j < 8; j++) ds[r][j] = h2f(dq[r][j]);
            }
        }
        load(ch + cs);
        f32x4 s[NT];
        scales(ch, s);
        const uint32_t so = ch * XF_CHUNK;
        SkX<NT> x[2];
        x[0].load(xr, xo, so, low);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (j < 7) x[(j + 1) & 1].load(xr, xo, so + (j + 1) * 2048, low);
            const SkX<NT>& X = x[j & 1];
#pragma unroll
            for (int r = 0; r < R; r++) {
                h8 hi, lo;
                float d;
                if constexpr (FMT == QP_F32) {
                    // the eight values scaled by a power of two of the largest among the row's 32
                    float v[8] = {__uint_as_float(c[r][2 * j][0]), __uint_as_float(c[r][2 * j][2]),
                                  __uint_as_float(c[r][2 * j][1]), __uint_as_float(c[r][2 * j][3]),
                                  __uint_as_float(c[r][2 * j + 1][0]), __uint_as_float(c[r][2 * j + 1][2]),
                                  __uint_as_float(c[r][2 * j + 1][1]), __uint_as_float(c[r][2 * j + 1][3])};
                    float mx = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
                    mx = fmaxf(mx, bfly_f<4>(mx, threadIdx.x & 63));
                    mx = fmaxf(mx, bfly_f<5>(mx, threadIdx.x & 63));
                    int e = (int)((__float_as_uint(mx) >> 23) & 255) - 127;
                    if (mx == 0.0f) e = 9;
                    if (e < -117) e = -117;
                    const float up = __uint_as_float((uint32_t)(9 - e + 127) << 23);
                    d = __uint_as_float((uint32_t)(e - 9 + 127) << 23);
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const float u = v[i] * up;
                        hi[i] = (_Float16)u;
                        const float rest = u - (float)hi[i];
                        lo[i] = (_Float16)(rest == rest ? rest : 0.0f);
                    }
                } else {
                    uint32_t a, b;  // bytes biased by 128: inputs 4g.. and 16 + 4g..
                    if constexpr (FMT == QP_Q8_0) {
                        a = c[r][j >> 1][(j & 1) * 2] ^ 0x80808080u;
                        b = c[r][j >> 1][(j & 1) * 2 + 1] ^ 0x80808080u;
                    } else {
                        const uint32_t q = c[r][j >> 2][j & 3];
                        a = iq4nl_lut4(q & 0x0f0f0f0fu) ^ 0x80808080u;
                        b = iq4nl_lut4((q >> 4) & 0x0f0f0f0fu) ^ 0x80808080u;
                    }
                    const h2 k14 = {(_Float16)16384.0f, (_Float16)16384.0f}, o = {(_Float16)-0.125f, (_Float16)-0.125f};
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t w8 = i < 2 ? a : b;
                        // byte * 2^-24 to (byte - 128) * 2^-10
                        const h2 v = __builtin_elementwise_fma(as_h2(((i & 1) ? w8 >> 8 : w8) & 0x00ff00ffu), k14, o);
                        hi[2 * i] = v[0];
                        hi[2 * i + 1] = v[1];
                    }
                    d = ds[r][j] * 0x1p10f;
                }
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    f32x4 p = sk_mfma(X.hi[t], hi, f32x4{0, 0, 0, 0});
                    p = sk_mfma(X.lo[t], hi, p);
                    if constexpr (FMT == QP_F32) p = sk_mfma(X.hi[t], lo, p);
#pragma unroll
                    for (int i = 0; i < 4; i++) tot[r][t][i] = fmaf(s[t][i], d * p[i], tot[r][t][i]);
                }
            }
        }
    }
}

// grid (row blocks, tpe slots of token blocks, times the experts), 256 threads: a.kw wavefronts (1, 2 or 4) take K slices
// of the same 16 R rows, 4 / a.kw row groups per workgroup; slot s takes the token blocks s, s + tpe, ... of 16 NT rows.
template <int FMT, int NT, int R>
QP_DEV void sk_body(const QpSkArgs& a) {
    constexpr bool KQ = FMT == QP_Q4_K || FMT == QP_Q5_K || FMT == QP_Q6_K || FMT == QP_Q3_K || FMT == QP_Q2_K;
    extern __shared__ float4 sk_lds[];
    __shared__ uint32_t jobs[16 * NT];
    f32x4* red = reinterpret_cast<f32x4*>(sk_lds);
    const uint32_t tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n16 = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (uniform: so are the resources made from it)
    uint32_t e = 0, o0 = 0, o1, slot = blockIdx.y;  // expert, its list entries (dense: the token rows)
    if (a.lst) {
        e = blockIdx.y / a.tpe;
        slot = blockIdx.y % a.tpe;
        o0 = __builtin_amdgcn_readfirstlane(gload<uint32_t>(a.off + 4ull * e));
        o1 = __builtin_amdgcn_readfirstlane(min(gload<uint32_t>(a.off + 4ull * e + 4), a.nlst));
    } else {
        o1 = pass_T(a.paso, a.tbase, a.rows);
    }
    const uint32_t nch = (a.k + 255) / 256, kw = wave % a.kw, rg = wave / a.kw;
    const uint32_t row0 = (blockIdx.x * (4 / a.kw) + rg) * 16 * R;
    const bool work = row0 < a.n;
    const uint32_t ntile = a.rows >> 4;
    const __amdgpu_buffer_rsrc_t xr = kq_rsrc(a.xs, (uint64_t)ntile * nch * XF_CHUNK);
    const __amdgpu_buffer_rsrc_t sr = kq_rsrc(a.xs + (uint64_t)ntile * nch * XF_CHUNK, (uint64_t)ntile * nch * 64);
    const bool dense = !a.lst;
    SkRows rw[R];
    if (work) {
        const uint64_t grow = (uint64_t)e * a.n + row0;  // first row in the tensor
        const uint64_t rest = a.wrows - grow;            // (the rows the tensor still holds: bounds the resource)
        uint64_t rb, db = 0;
        if constexpr (KQ) {
            rb = (uint64_t)nch * SkK<FMT>::RB;
            if constexpr (FMT == QP_Q6_K) db = nch * 2ull;
            if constexpr (FMT == QP_Q2_K) db = nch * 4ull;
        } else {
            rb = FMT == QP_F32 ? 4ull * a.k : FMT == QP_Q8_0 ? a.k : a.k / 2;
            db = FMT == QP_F32 ? 0 : a.k / 32 * 2ull;
        }
        const uint64_t hold = rest < 16 * R ? rest : 16 * R;
        const __amdgpu_buffer_rsrc_t wr = kq_rsrc(a.w + grow * rb, hold * rb);
        const __amdgpu_buffer_rsrc_t dr = kq_rsrc(a.w + a.wrows * rb + grow * db, hold * db);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t rr = r * 16 + n16;
            rw[r].w = wr;
            rw[r].d = dr;
            rw[r].off = row0 + rr < a.n ? rr * (uint32_t)rb : QP_NOOFF;
            rw[r].doff = rr * (uint32_t)db;
        }
    }
    const uint32_t per = KQ ? 4 : 1, units = (nch + per - 1) / per;
    for (uint32_t t0 = o0 + slot * (16 * NT); t0 < o1; t0 += a.tpe * (16 * NT)) {
        const uint32_t cnt = min(o1 - t0, 16u * NT);  // rows of this block
        if (!dense) {
            if (tid < 16 * NT) {
                uint32_t j = tid < cnt ? gload<uint32_t>(a.lst + 4ull * (t0 + tid)) : QP_NOOFF;
                if (j != QP_NOOFF && (j >= a.yrows || j / a.tfijo >= a.xrows)) j = QP_NOOFF;
                jobs[tid] = j;
            }
            __syncthreads();
        }
        // X: per lane the operand row of each token tile (dense: the tile's own lane), and the rows' scales
        uint32_t xo[NT], so[NT][4];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (dense) {
                const bool in = (uint32_t)t * 16 < cnt;  // (the tile's rows past T are zeros)
                xo[t] = in ? xf_tile(t0 + t * 16, nch) + lane * 16 : QP_NOOFF;
                so[t][0] = in ? ((t0 >> 4) + t) * nch * 64 + g * 16 : QP_NOOFF;
            } else {
                const uint32_t j = jobs[t * 16 + n16];
                xo[t] = j == QP_NOOFF ? QP_NOOFF : xf_tile(j / a.tfijo, nch) + ((j / a.tfijo) & 15) * 128 + g * 16;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t ji = jobs[t * 16 + 4 * g + i], x = ji / a.tfijo;
                    so[t][i] = ji == QP_NOOFF ? QP_NOOFF : (x >> 4) * nch * 64 + (x & 15) * 4;
                }
            }
        }
        auto scales = [&](uint32_t ch, f32x4(&s)[NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if (dense) {
                    s[t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(sr, so[t][0], ch * 64, 0));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        s[t][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sr, so[t][i], ch * 64, 0));
                }
            }
        };
        f32x4 tot[R][NT];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int t = 0; t < NT; t++) tot[r][t] = f32x4{0, 0, 0, 0};
        if (work && kw < units) {
            if constexpr (KQ) sk_kq<FMT, NT, R>(rw, nch, kw, units, a.kw, xr, xo, dense ? 1024 : XF_LOW, scales, tot);
            else sk_pl<FMT, NT, R>(rw, a.k, kw, units, a.kw, xr, xo, dense ? 1024 : XF_LOW, scales, tot);
        }
        // the K slices' sums, added in their order; wavefront kw of a row group finishes its share of the tiles
        if (a.kw > 1) {
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int t = 0; t < NT; t++) red[(wave * R * NT + r * NT + t) * 64 + lane] = tot[r][t];
            __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint32_t at = r * NT + t, n = row0 + r * 16 + n16;
                if (at % a.kw != kw || n >= a.n) continue;
                f32x4 v = tot[r][t];
                if (a.kw > 1) {
                    v = red[(rg * a.kw * R * NT + at) * 64 + lane];
                    for (uint32_t q = 1; q < a.kw; q++) v += red[((rg * a.kw + q) * R * NT + at) * 64 + lane];
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t m = t * 16 + 4 * g + i;
                    if (m >= cnt) continue;
                    uint32_t yr = t0 + m;
                    if (!dense) {
                        yr = jobs[m];
                        if (yr == QP_NOOFF) continue;
                    }
                    const uint64_t at_y = a.y + 4 * ((uint64_t)yr * a.n + n);
                    gstore<float>(at_y, a.acc ? gload<float>(at_y) + v[i] : v[i]);
                }
            }
        if (t0 + a.tpe * (16 * NT) < o1) __syncthreads();  // the jobs and sums are read before the next block's
    }
}

#define SK_KERNEL(NAME, FMT, NT, R)                                                                                 \
    KERNEL __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NT * R == 8 ? 1 : 2))) void                    \
    qp_sk_##NAME##_t##NT##r##R(QpSkArgs a) {                                                                        \
        sk_body<FMT, NT, R>(a);                                                                                     \
    }
#define SK_KERNELS(NAME, FMT, R) SK_KERNEL(NAME, FMT, 1, R) SK_KERNEL(NAME, FMT, 2, R) SK_KERNEL(NAME, FMT, 4, R)
SK_KERNELS(q4k, QP_Q4_K, 1) SK_KERNELS(q4k, QP_Q4_K, 2)
SK_KERNELS(q5k, QP_Q5_K, 1) SK_KERNELS(q5k, QP_Q5_K, 2)
SK_KERNELS(q6k, QP_Q6_K, 1) SK_KERNELS(q6k, QP_Q6_K, 2)
SK_KERNELS(q3k, QP_Q3_K, 1) SK_KERNELS(q3k, QP_Q3_K, 2)
SK_KERNELS(q2k, QP_Q2_K, 1) SK_KERNELS(q2k, QP_Q2_K, 2)
SK_KERNELS(q8, QP_Q8_0, 1)
SK_KERNELS(iq4nl, QP_IQ4_NL, 1)
SK_KERNELS(f32, QP_F32, 1)
SK_KERNEL(f32, QP_F32, 4, 2)
