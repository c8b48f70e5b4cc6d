// Weights as integers times f32 scales, and X as f16 operands, for the matrix-core matmuls (qp_small.hip, qp_tile.hip).
#pragma once
#include "qp_common.h"

#define KERNEL extern "C" __global__

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// X as operands: for each tile of 16 rows and chunk of 256 inputs, 8 steps of 32 inputs, 2 KB each, then the operand of
// the chunk's 16 sums of 16 inputs (lane groups 0, 1: their high parts, 2, 3: low parts).  Lane g * 16 + m of step j holds
// row m's inputs 32 j + {4g, 4g + 2, 4g + 1, 4g + 3, 16 + 4g, 18 + 4g, 17 + 4g, 19 + 4g} as 16 bytes of high parts and
// 16 of low ones.  Dense matmuls read whole tiles: the 64 lanes' high parts and then the low ones, lane after lane.
// Grouped ones gather rows: row m's 128 bytes of a step (four lanes' high parts, then the low ones) are one cache line
// (with the dense order a gathered 16 bytes took a line each: MoE FFN of 128 Q4_K experts 768 x 2048 at 2048 tokens 1722
// us, 869 with this one; the dense matmul of 32 tokens the other way round, 8B layer: 291 us in this order, 171 in its own).
// The chunks' scales (one float per row and chunk: the stored values times it are X) follow all tiles.
constexpr uint32_t XF_CHUNK = 18 * 1024;  // bytes of a tile's chunk
constexpr uint32_t XF_LOW = 64;           // grouped: from a lane's high parts to its low ones (dense: 1024)

QP_DEV uint32_t xf_tile(uint32_t row, uint32_t nch) { return (row >> 4) * nch * XF_CHUNK; }

QP_DEV h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }

// Two bytes of w as f16 times 2^-SH (-5 <= SH <= 6) plus off * 2^-SH: the byte in the low mantissa bits
// of a power of two (1024 at SH = 0), which the addition takes away.
template <int SH>
QP_DEV h2 sk_dup(uint32_t w, uint32_t sel, float off = 0.0f) {
    constexpr uint32_t top = 0x64u - SH * 4;  // high byte of 2^(10 - SH)
    constexpr float unit = SH >= 0 ? 1.0f / (1 << (SH > 0 ? SH : 0)) : (float)(1 << (SH < 0 ? -SH : 0));
    const float c = (off - 1024.0f) * unit;
    const h2 o = {(_Float16)c, (_Float16)c};
    return as_h2(__builtin_amdgcn_perm(top * 0x01010101u, w, sel)) + o;
}
constexpr uint32_t sk_sel(int i, int j) { return 0x04000400u | (uint32_t)i | ((uint32_t)j << 16); }

// The quants stay where they are in the low 10 bits of a half, which as f16 is a subnormal: value * 2^-24 times the
// power of two of their position (exact).  The scale they are multiplied by takes the position's power away and carries
// 32 times the power of two SkK::UP, so that the products are normal f16: the matrix instructions take subnormal
// operands, but align them as if their leading bit were set, and drop the low bits of the sum (Q2_K 4e-6 off instead of
// 3e-7 at K = 1024).  The block's f32 scale takes all of it away.

// ------------------------------------------------------------------ K-quants
template <int FMT> struct SkK;
template <> struct SkK<QP_Q4_K> { static constexpr int NC = 9, HDR = 0, RB = 144, UP = 2; static constexpr bool MIN = true, LO = false; };
template <> struct SkK<QP_Q5_K> { static constexpr int NC = 11, HDR = 0, RB = 176, UP = 2; static constexpr bool MIN = true, LO = false; };
template <> struct SkK<QP_Q6_K> { static constexpr int NC = 13, HDR = 12, RB = 208, UP = 0; static constexpr bool MIN = true, LO = true; };
template <> struct SkK<QP_Q3_K> { static constexpr int NC = 7, HDR = 6, RB = 112, UP = 2; static constexpr bool MIN = false, LO = false; };
template <> struct SkK<QP_Q2_K> { static constexpr int NC = 5, HDR = 0, RB = 80, UP = 4; static constexpr bool MIN = true, LO = false; };

// Scales and minima of a block, from its header chunk h (and dd: Q6_K: d, Q2_K: d, dmin, the arrays after the rows).
// The block is d * 2^(19 - UP) * sum(products of sk_quad) - dmin * sum(mins * sums of 16 inputs).
template <int FMT>
struct SkScales {
    uint32_t h[4], dd;
    uint32_t sc[4];   // scales times 2^UP: Q4_K/Q5_K sub-blocks 0..7 in sc[0..1] (minima in sc[2..3]); others 16 bytes

    QP_DEV void setup() {
        if constexpr (FMT == QP_Q4_K || FMT == QP_Q5_K) {
            sc[0] = (h[1] << 2) & 0xfcfcfcfcu;
            sc[1] = ((h[3] << 2) & 0x3c3c3c3cu) | (h[1] & 0xc0c0c0c0u);
            sc[2] = h[2] & 0x3f3f3f3fu;
            sc[3] = ((h[3] >> 4) & 0x0f0f0f0fu) | ((h[2] >> 2) & 0x30303030u);
        } else if constexpr (FMT == QP_Q6_K) {
#pragma unroll
            for (int i = 0; i < 4; i++) sc[i] = h[i] ^ 0x80808080u;
        } else if constexpr (FMT == QP_Q3_K) {
            const uint32_t k1 = 0xc0c0c0c0u, k2 = 0x3c3c3c3cu;
            sc[0] = ((h[0] << 2) & k2) | ((h[2] << 6) & k1);
            sc[1] = ((h[1] << 2) & k2) | ((h[2] << 4) & k1);
            sc[2] = ((h[0] >> 2) & k2) | ((h[2] << 2) & k1);
            sc[3] = ((h[1] >> 2) & k2) | (h[2] & k1);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) sc[i] = (h[i] << 4) & 0xf0f0f0f0u;
        }
    }
    QP_DEV float d() const {
        if constexpr (FMT == QP_Q4_K || FMT == QP_Q5_K) return h2f(h[0]);
        else if constexpr (FMT == QP_Q3_K) return h2f(h[3]);
        else return h2f(dd);
    }
    QP_DEV float dmin() const {
        if constexpr (FMT == QP_Q4_K || FMT == QP_Q5_K) return h2f(h[0] >> 16);
        else if constexpr (FMT == QP_Q2_K) return h2f(dd >> 16);
        else return h2f(dd);  // Q6_K: d * 32 * scale is taken from every input
    }
    // The minima's operand: lane groups 0 and 2: of the first eight sums of 16 inputs, 1 and 3: of the others.
    QP_DEV h8 mins(uint32_t g) const {
        h2 v[4];
        if constexpr (FMT == QP_Q4_K || FMT == QP_Q5_K) {
            const uint32_t m = (g & 1) ? sc[3] : sc[2];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = sk_dup<0>(m, sk_sel(i, i));
        } else {
            const uint32_t a = (g & 1) ? (FMT == QP_Q6_K ? sc[2] : h[2]) : (FMT == QP_Q6_K ? sc[0] : h[0]);
            const uint32_t b = (g & 1) ? (FMT == QP_Q6_K ? sc[3] : h[3]) : (FMT == QP_Q6_K ? sc[1] : h[1]);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t w = i < 2 ? a : b, sel = sk_sel(2 * (i & 1), 2 * (i & 1) + 1);
                if constexpr (FMT == QP_Q6_K) v[i] = sk_dup<-5>(w, sel, -128.0f);  // 32 times the scale
                else v[i] = sk_dup<0>((w >> 4) & 0x0f0f0f0fu, sel);
            }
        }
        h8 r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r[2 * i] = v[i][0];
            r[2 * i + 1] = v[i][1];
        }
        return r;
    }
    // The f16 scale of the first (i = 0) or second 16 inputs of step j (32 inputs), for quants at bit AT of their halves.
    template <int j, int AT>
    QP_DEV h2 scale(int i) const {
        if constexpr (FMT == QP_Q4_K || FMT == QP_Q5_K) return sk_dup<AT - 5>(sc[j >> 2], sk_sel(j & 3, j & 3));
        else return sk_dup<AT - 5>(sc[(2 * j + i) >> 2], sk_sel((2 * j + i) & 3, (2 * j + i) & 3),
                                   FMT == QP_Q2_K ? 0.0f : -128.0f);
    }
};

// Where step j's quants are: data chunk of its first 16 inputs (the second 16: the next chunk), the bit AT of their
// bytes, and the chunk of the high bits (-1: none) with the shift UP that takes them to their place.
template <int FMT, int j>
struct SkStep {
    static constexpr int CHUNK = FMT == QP_Q4_K ? 1 + 2 * (j >> 1) : FMT == QP_Q5_K ? 3 + 2 * (j >> 1)
                               : FMT == QP_Q6_K ? 4 * (j >> 2) + (j & 1) * 2 : FMT == QP_Q3_K ? 2 + 2 * (j >> 2) : 1 + 2 * (j >> 2);
    static constexpr int AT = FMT == QP_Q4_K || FMT == QP_Q5_K ? (j & 1) * 4 : FMT == QP_Q6_K ? ((j >> 1) & 1) * 4 : 2 * (j & 3);
    static constexpr int HIGH = FMT == QP_Q5_K ? 1 : FMT == QP_Q6_K ? 8 + 2 * (j >> 2) : FMT == QP_Q3_K ? 0 : -1;
    static constexpr int UP = FMT == QP_Q5_K ? 4 + AT - j : FMT == QP_Q6_K ? 4 + AT - 2 * (j & 3) : 2 + AT - j;
};

// scale * quant * 2^(UP - 19) of the four bytes of w (high bits from hb) as f16, in the order 0, 2, 1, 3; lo: what is left
// of Q6_K's products, which reach 8064.
template <int FMT, int j>
QP_DEV void sk_quad(uint32_t w, uint32_t hb, h2 s, h2 (&q)[2], h2 (&lo)[2]) {
    using S = SkStep<FMT, j>;
    constexpr int at = S::AT, up = S::UP;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        constexpr uint32_t mask = FMT == QP_Q3_K || FMT == QP_Q2_K ? 0x00030003u : 0x000f000fu;
        uint32_t v = (i ? w >> 8 : w) & (mask << at);
        if constexpr (S::HIGH >= 0) {
            constexpr uint32_t hm = FMT == QP_Q5_K ? 0x00100010u : FMT == QP_Q6_K ? 0x00300030u : 0x00040004u;
            const uint32_t x = i ? (up >= 8 ? hb << (up >= 8 ? up - 8 : 0) : hb >> (up >= 8 ? 0 : 8 - up))
                                 : (up >= 0 ? hb << (up >= 0 ? up : 0) : hb >> (up >= 0 ? 0 : -up));
            v |= x & (hm << at);
        }
        if constexpr (FMT == QP_Q3_K) {
            constexpr float m4 = -4.0f * (1 << at) * 0x1p-24f;
            q[i] = __builtin_elementwise_fma(as_h2(v), s, s * h2{(_Float16)m4, (_Float16)m4});  // (q - 4) scale, exact
        } else {
            q[i] = as_h2(v) * s;
            if constexpr (FMT == QP_Q6_K) lo[i] = __builtin_elementwise_fma(as_h2(v), s, -q[i]);
        }
    }
}

QP_DEV f32x4 sk_mfma(h8 a, h8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

template <int V> struct SkInt { static constexpr int v = V; };
