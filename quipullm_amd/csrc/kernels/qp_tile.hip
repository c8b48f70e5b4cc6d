// K-quant matrix products of many token rows (matmul_<fmt>_t, matmul_<fmt>_t_swiglu, matmul_<fmt>_eg with many jobs per
// expert) on integer weights (qp_ints.h), in tiles of 128 token rows x 128 weight rows.
//
// Four wavefronts of 64 x 64 (2 x 2 instructions of 32 x 32 x 16, two accumulators each: the block's integer sums and the
// total).  Per step of 32 inputs every thread turns 16 weights of one row into their operands (scale * quant as f16: a
// mask and a multiplication per two weights) and copies 64 bytes of X's operands (qp_split_f16), both into the LDS
// buffer that the next step reads; the loads of the step after are in flight meanwhile.  Every 256 inputs the integer
// sums are scaled by the block's f32 scale and the row's, less the minima times X's sums of 16 inputs (two instructions
// per 32 x 32).  64 KB of LDS (80 KB for Q6_K): two workgroups per CU, whose barriers overlap.
//
// Bound by no unit alone: every weight takes two instructions' worth of products (X's two halves; Q6_K three), and in Q4_K
// 14336 x 4096 at 2048 tokens the matrix cores are busy 49 % of the cycles and LDS 50 %, of which a quarter is bank conflicts,
// at a clock that the load has brought to 1.9 GHz, and the wavefronts wait 26 % of theirs; Q6_K 4096 x 14336 50 / 44 / 29 % at
// 1.7 GHz, at 256 tokens (7 blocks per K split, the inputs from farther away) 30 / 26 / 38 % at 2.2.
// Measured in us, in parentheses 256-token tiles of bf16 planes of both sides (three products): Q4_K 14336 x 4096 at 2048 tokens
// 519 with the input's split (629), 0.93 PFLOP/s of f16 products, where the library's dense f16 product reaches 1.15 to 1.2; Q6_K
// 4096 x 14336 770 (781).  With the staging left out 0.88 of the time; with instructions of 16 x 16 x 32 1.07 of it.
#include "qp_ints.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
QP_DEV f32x16 tl_mfma(h8 a, h8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

// sums over a wavefront, and up to each lane
QP_DEV uint32_t wave_scan_u(uint32_t v, uint32_t lane) {
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
        const uint32_t u = __shfl_up(v, k, 64);
        if (lane >= (uint32_t)k) v += u;
    }
    return v;
}
QP_DEV uint32_t wave_sum_u(uint32_t v) {
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) v += __shfl_xor(v, k, 64);
    return __builtin_amdgcn_readfirstlane(v);
}

// LDS bytes of 16 token rows' operands: their 16-byte pieces in the order of the lanes, 16 bytes of room after each lane
// group, so that the eight pieces of a row that consecutive threads write lie in different banks
constexpr uint32_t XG = 272, XP = 4 * XG, XT = 2 * XP;

template <int FMT, bool GLU>
QP_DEV void tile_body(const QpTileArgs& a) {
    using F = SkK<FMT>;
    constexpr uint32_t XB = 8 * XT, WB = F::LO ? 16384 : 8192;
    constexpr int ND = FMT == QP_Q3_K || FMT == QP_Q2_K ? 2 : 4;             // data chunks of a thread per block
    constexpr int NH = FMT == QP_Q6_K ? 2 : FMT == QP_Q5_K || FMT == QP_Q3_K ? 1 : 0;  // high-bit chunks
    extern __shared__ float4 tl_lds[];
    char* const lds = reinterpret_cast<char*>(tl_lds);
    char* const xb = lds;                    // [2][8 tiles][high, low][4 lane groups][16 rows of 16, room]
    char* const wb = lds + 2 * XB;           // [2][(Q6_K: high, low)][8 row tiles][64 lanes][16]
    char* const sums = wb + 2 * WB;          // [8 tiles][64 lanes][16]
    char* const mins = sums + 8192;          // [128 rows][32]
    float* const dd = reinterpret_cast<float*>(mins + 4096);  // [128 rows] d, then [128] dmin
    float* const scl = dd + 256;             // [128 token rows]
    __shared__ uint32_t jobs[128];
    const uint32_t tid = threadIdx.x, lane = tid & 63, n16 = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    // ---- this workgroup's tile: consecutive ones on the same XCD (workgroup id % 8)
    uint32_t e = 0, t0, cnt, nti;
    const bool dense = GLU || !a.lst;
    const uint32_t in_xcd = blockIdx.x >> 3;
    if (dense) {  // eight row tiles at a time
        const uint32_t parts = 8 / a.zx, total = a.mt * a.nt, chunk = (total + parts - 1) / parts;
        const uint32_t L = (blockIdx.x & 7) / a.zx * chunk + in_xcd;
        if (in_xcd >= chunk || L >= total) return;
        const uint32_t grp = L / (a.mt * 8), rem = L % (a.mt * 8), in = min(8u, a.nt - grp * 8);
        t0 = (rem / in) * 128;
        nti = grp * 8 + rem % in;
        const uint32_t T = pass_T(a.paso, a.tbase, a.rows);
        if (t0 >= T) return;
        cnt = min(T - t0, 128u);
    } else {  // the experts' 128-job tiles that are there, in order: the experts' counts scanned by every wavefront
        auto tiles = [&](uint32_t x) -> uint32_t {  // (0 past the last expert)
            if (x >= a.nexp) return 0;
            const uint32_t o0 = gload<uint32_t>(a.off + 4ull * x), o1 = min(gload<uint32_t>(a.off + 4ull * x + 4), a.nlst);
            const uint32_t n = o1 > o0 ? o1 - o0 : 0;
            return (n + 127) / 128;
        };
        uint32_t nslot = 0;
        for (uint32_t x0 = 0; x0 < a.nexp; x0 += 64) nslot += wave_sum_u(tiles(x0 + lane));
        const uint32_t total = nslot * a.nt, chunk = (total + 7) / 8, L = (blockIdx.x & 7) * chunk + in_xcd;
        if (in_xcd >= chunk || L >= total) return;
        const uint32_t s = L / a.nt;
        nti = L % a.nt;
        uint32_t done = 0, slot = 0;
        for (uint32_t x0 = 0; x0 < a.nexp; x0 += 64) {
            const uint32_t c = tiles(x0 + lane);
            const uint32_t incl = done + wave_scan_u(c, lane);
            const uint64_t hit = __ballot(incl > s);
            if (hit) {
                const int l = __builtin_ctzll(hit);
                e = x0 + l;
                slot = s - (__builtin_amdgcn_readlane(incl, l) - __builtin_amdgcn_readlane(c, l));
                break;
            }
            done = __builtin_amdgcn_readlane(incl, 63);
        }
        e = __builtin_amdgcn_readfirstlane(e);
        const uint32_t o0 = __builtin_amdgcn_readfirstlane(gload<uint32_t>(a.off + 4ull * e));
        const uint32_t o1 = __builtin_amdgcn_readfirstlane(min(gload<uint32_t>(a.off + 4ull * e + 4), a.nlst));
        t0 = o0 + slot * 128;
        if (t0 >= o1) return;
        cnt = min(o1 - t0, 128u);
        if (tid < 128) {
            uint32_t j = tid < cnt ? gload<uint32_t>(a.lst + 4ull * (t0 + tid)) : QP_NOOFF;
            if (j != QP_NOOFF && (j >= a.yrows || j / a.tfijo >= a.xrows)) j = QP_NOOFF;
            jobs[tid] = j;
        }
        __syncthreads();
    }
    const uint32_t n0 = nti * (GLU ? 64 : 128), nb = a.k / 256;
    // ---- staging: row rr of the tile, half hf of each 32 inputs; X: 16 bytes of tile q * 2 + tid / 128, plane, lane
    const uint32_t rr = tid >> 1, hf = tid & 1;
    const uint32_t lrow = GLU ? rr & 63 : rr;
    const uint64_t rb = (uint64_t)nb * F::RB, db = FMT == QP_Q6_K ? nb * 2ull : FMT == QP_Q2_K ? nb * 4ull : 0;
    const uint64_t grow = (uint64_t)e * a.n + n0, rest = a.wrows - grow, hold = rest < (GLU ? 64 : 128) ? rest : (GLU ? 64 : 128);
    const uint64_t wbase = GLU && wave >= 2 ? a.w2 : a.w;
    const __amdgpu_buffer_rsrc_t wr = kq_rsrc(wbase + grow * rb, hold * rb), dr = kq_rsrc(wbase + a.wrows * rb + grow * db, hold * db);
    const uint32_t roff = n0 + lrow < a.n ? lrow * (uint32_t)rb : QP_NOOFF;
    const uint32_t rofh = roff == QP_NOOFF ? QP_NOOFF : roff + hf * nb * 16;
    const uint32_t rofd = roff == QP_NOOFF ? QP_NOOFF : lrow * (uint32_t)db;
    const uint32_t ntile = a.rows >> 4;
    const __amdgpu_buffer_rsrc_t xr = kq_rsrc(a.xs, (uint64_t)ntile * nb * XF_CHUNK);
    const __amdgpu_buffer_rsrc_t sr = kq_rsrc(a.xs + (uint64_t)ntile * nb * XF_CHUNK, (uint64_t)ntile * nb * 64);
    // offset of piece (plane, lane group) of tile row m's operands (chunk 0)
    auto xrow = [&](uint32_t m, uint32_t plane, uint32_t g) -> uint32_t {
        if (dense) return m < cnt ? xf_tile(t0 + m, nb) + plane * 1024 + g * 256 + (m & 15) * 16 : QP_NOOFF;
        const uint32_t x = jobs[m] / a.tfijo;
        return jobs[m] == QP_NOOFF ? QP_NOOFF : xf_tile(x, nb) + (x & 15) * 128 + plane * XF_LOW + g * 16;
    };
    // X: 16-byte pieces so that consecutive threads read consecutive ones
    const uint32_t xg = dense ? (tid >> 4) & 3 : tid & 3, xp = dense ? (tid >> 6) & 1 : (tid >> 2) & 1;
    const uint32_t xm = dense ? (tid >> 7) * 16 + n16 : tid >> 3;
    uint32_t xo[4], so[2];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        xo[q] = xrow(q * 32 + xm, xp, xg);
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const uint32_t at = q * 256 + tid, o = xrow((at >> 6) * 16 + (at & 15), 0, (at >> 4) & 3);
        so[q] = o == QP_NOOFF ? QP_NOOFF : o + 16384;
    }
    char* const xst = xb + (xm >> 4) * XT + xp * XP + xg * XG + (xm & 15) * 16;
    uint32_t co = QP_NOOFF;  // this thread's token row's scale
    if (tid < 128) {
        const uint32_t x = dense ? t0 + tid : jobs[tid] == QP_NOOFF ? 0 : jobs[tid] / a.tfijo;
        if (dense ? tid < cnt : jobs[tid] != QP_NOOFF) co = (x >> 4) * nb * 64 + (x & 15) * 4;
    }
    const uint32_t split = a.zx > 1 ? (blockIdx.x & 7) % a.zx : blockIdx.z;
    const uint32_t b0 = split * a.kb, b1 = min(nb, b0 + a.kb);

    u32x4 D[ND], H[NH > 0 ? NH : 1], hn;
    uint32_t ddn = 0;
    SkScales<FMT> sc;
    u32x4 xv[4], sv[2];
    float cv = 0.0f;
    auto load_d = [&](int i, uint32_t blk) __attribute__((always_inline)) {
        const int c = FMT == QP_Q4_K ? 1 + 2 * i : FMT == QP_Q5_K ? 3 + 2 * i : FMT == QP_Q6_K ? 2 * i : FMT == QP_Q3_K ? 2 + 2 * i : 1 + 2 * i;
        D[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, rofh, (c * nb + blk) * 16, 0);
    };
    auto load_h = [&](int i, uint32_t blk) __attribute__((always_inline)) {
        const int c = FMT == QP_Q5_K ? 1 : FMT == QP_Q6_K ? 8 + 2 * i : 0;
        H[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, rofh, (c * nb + blk) * 16, 0);
    };
    auto load_hdr = [&](uint32_t blk) __attribute__((always_inline)) {
        hn = __builtin_amdgcn_raw_buffer_load_b128(wr, roff, (F::HDR * nb + blk) * 16, 0);
        if constexpr (FMT == QP_Q6_K) ddn = __builtin_amdgcn_raw_buffer_load_b16(dr, rofd, blk * 2, 0);
        if constexpr (FMT == QP_Q2_K) ddn = __builtin_amdgcn_raw_buffer_load_b32(dr, rofd, blk * 4, 0);
    };
    auto load_x = [&](uint32_t blk, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; q++) xv[q] = __builtin_amdgcn_raw_buffer_load_b128(xr, xo[q], blk * XF_CHUNK + j * 2048, 0);
    };
    auto take_hdr = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) sc.h[i] = hn[i];
        sc.dd = ddn;
        sc.setup();
    };
    // step j of the thread's block to LDS buffer buf, then the next block's loads into the registers that are done with
    auto stage = [&](auto J, int buf, uint32_t next) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::v;
        using S = SkStep<FMT, j>;
        constexpr int di = FMT == QP_Q4_K || FMT == QP_Q5_K ? j >> 1 : FMT == QP_Q6_K ? (j >> 2) * 2 + (j & 1) : j >> 2;
        constexpr int hi = FMT == QP_Q6_K ? j >> 2 : 0;
        const h2 s0 = sc.template scale<j, S::AT>(0), s1 = sc.template scale<j, S::AT>(1);
        const h2 s = FMT == QP_Q4_K || FMT == QP_Q5_K ? s0 : as_h2(hf ? __builtin_bit_cast(uint32_t, s1) : __builtin_bit_cast(uint32_t, s0));
        char* const w = wb + buf * WB + (rr >> 4) * 1024 + (rr & 15) * 16 + hf * 8;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            h2 q[2], l[2];
            sk_quad<FMT, j>(D[di][k], NH > 0 ? H[hi][k] : 0u, s, q, l);
            *reinterpret_cast<uint2*>(w + k * 256) = make_uint2(__builtin_bit_cast(uint32_t, q[0]), __builtin_bit_cast(uint32_t, q[1]));
            if constexpr (F::LO)
                *reinterpret_cast<uint2*>(w + 8192 + k * 256) = make_uint2(__builtin_bit_cast(uint32_t, l[0]), __builtin_bit_cast(uint32_t, l[1]));
        }
#pragma unroll
        for (int q = 0; q < 4; q++) *reinterpret_cast<u32x4*>(xst + buf * XB + q * 2 * XT) = xv[q];
        constexpr bool dlast = FMT == QP_Q4_K || FMT == QP_Q5_K ? j & 1 : FMT == QP_Q6_K ? (j & 2) != 0 : (j & 3) == 3;
        constexpr bool hlast = FMT == QP_Q6_K ? (j & 3) == 3 : j == 7;
        if constexpr (dlast) load_d(di, next);
        if constexpr (NH > 0 && hlast) load_h(hi, next);
    };
    f32x16 p[2][2], tot[2][2];  // [row block of 32][token block of 32]
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int t = 0; t < 2; t++) tot[r][t] = f32x16{};
    // this lane's 16 bytes of a pair of 16-row operands as one of 32 rows and 16 inputs (the first or second lane groups)
    const uint32_t fo = lane >> 5, f16o = ((lane >> 4) & 1), fl = (fo * 16 + n16) * 16;
    auto compute = [&](auto J, int buf) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::v;
        const char* const x = xb + buf * XB + wm * 4 * XT + f16o * XT + fo * XG + n16 * 16;
        const char* const w = wb + buf * WB + wn * 4096 + f16o * 1024 + fl;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            h8 b[2], l[2], xh[2], xl[2];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                b[r] = *reinterpret_cast<const h8*>(w + r * 2048 + h * 512);
                if constexpr (F::LO) l[r] = *reinterpret_cast<const h8*>(w + 8192 + r * 2048 + h * 512);
            }
#pragma unroll
            for (int t = 0; t < 2; t++) {
                xh[t] = *reinterpret_cast<const h8*>(x + t * 2 * XT + h * 2 * XG);
                xl[t] = *reinterpret_cast<const h8*>(x + t * 2 * XT + XP + h * 2 * XG);
            }
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 2; r++) p[r][t] = tl_mfma(xh[t], b[r], j || h ? p[r][t] : f32x16{});
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 2; r++) p[r][t] = tl_mfma(xl[t], b[r], p[r][t]);
            if constexpr (F::LO) {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int r = 0; r < 2; r++) p[r][t] = tl_mfma(xh[t], l[r], p[r][t]);
            }
        }
    };
    if (b0 < b1) {
        load_hdr(b0);
#pragma unroll
        for (int i = 0; i < ND; i++) load_d(i, b0);
#pragma unroll
        for (int i = 0; i < NH; i++) load_h(i, b0);
        load_x(b0, 0);
        take_hdr();
        stage(SkInt<0>(), 0, min(b0 + 1, b1 - 1));
        load_x(b0, 1);
        __syncthreads();
        auto loop = [&](auto LIVE) __attribute__((always_inline)) {
            for (uint32_t blk = b0; blk < b1; blk++) {
                const uint32_t next = min(blk + 1, b1 - 1);
                auto step = [&](auto J) __attribute__((always_inline)) {
                    constexpr int j = decltype(J)::v;
                    if constexpr (LIVE.v) compute(J, j & 1);
                    if constexpr (j == 0) {  // the block's minima and scales, and X's sums and scales: read after its last step
                        if constexpr (F::MIN) {
#pragma unroll
                            for (int q = 0; q < 2; q++) sv[q] = __builtin_amdgcn_raw_buffer_load_b128(xr, so[q], blk * XF_CHUNK, 0);
                            *reinterpret_cast<h8*>(mins + rr * 32 + hf * 16) = sc.mins(hf);
                        }
                        cv = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(sr, co, blk * 64, 0));
                        dd[hf * 128 + rr] = hf ? sc.dmin() : sc.d() * (float)(1 << (19 - F::UP));
                    }
                    if constexpr (j == 1) {
                        if constexpr (F::MIN) {
#pragma unroll
                            for (int q = 0; q < 2; q++) *reinterpret_cast<u32x4*>(sums + (q * 256 + tid) * 16) = sv[q];
                        }
                        if (tid < 128) scl[tid] = cv;
                    }
                    if constexpr (j == 3) load_hdr(next);
                    if constexpr (j < 7) stage(SkInt<(j + 1) & 7>(), (j + 1) & 1, next);
                    else {
                        // the block's sums into the totals
#pragma unroll
                        for (int r = 0; r < (LIVE.v ? 2 : 0); r++) {
                            const uint32_t row = wn * 64 + r * 32 + (lane & 31);
                            const float d = dd[row], dm = dd[128 + row];
                            h8 mn;
                            if constexpr (F::MIN) mn = *reinterpret_cast<const h8*>(mins + row * 32 + fo * 16);
#pragma unroll
                            for (int t = 0; t < 2; t++) {
                                f32x16 m;
                                if constexpr (F::MIN) {
                                    const char* const sx = sums + (wm * 4 + t * 2 + f16o) * 1024 + fl;
                                    m = tl_mfma(*reinterpret_cast<const h8*>(sx), mn, f32x16{});
                                    m = tl_mfma(*reinterpret_cast<const h8*>(sx + 512), mn, m);
                                }
#pragma unroll
                                for (int q = 0; q < 4; q++) {
                                    const f32x4 s = *reinterpret_cast<const f32x4*>(scl + wm * 64 + t * 32 + 8 * q + 4 * fo);
#pragma unroll
                                    for (int i = 0; i < 4; i++) {
                                        const int v = 4 * q + i;
                                        const float u = F::MIN ? fmaf(d, p[r][t][v], -(dm * m[v])) : d * p[r][t][v];
                                        tot[r][t][v] = fmaf(s[i], u, tot[r][t][v]);
                                    }
                                }
                            }
                        }
                        take_hdr();
                        stage(SkInt<0>(), 0, min(blk + 2, b1 - 1));
                    }
                    if constexpr (j < 6) load_x(blk, j + 2);
                    else load_x(next, j - 6);
                    __syncthreads();
                };
                step(SkInt<0>()); step(SkInt<1>()); step(SkInt<2>()); step(SkInt<3>());
                step(SkInt<4>()); step(SkInt<5>()); step(SkInt<6>()); step(SkInt<7>());
            }
        };
        if (GLU || wm * 64 < cnt) loop(SkInt<1>());  // (else the wavefront's token rows are all past the end)
        else loop(SkInt<0>());
    }
    if constexpr (GLU) {
        // silu(gate) * up: the up wavefronts' totals through LDS ([wm][row tile][token tile][lane]), the gate
        // wavefronts' results to f32 rows, or through an LDS tile [128 tokens][64 outputs] to the next matmul's input
        // planes (qp_split_bf16's values and layout)
        float* const ex = reinterpret_cast<float*>(lds);  // 32 KB (the last step's barrier is past)
        if (wn == 1) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) ex[(((wm * 2 + r) * 2 + t) * 16 + v) * 64 + lane] = tot[r][t][v];
        }
        __syncthreads();
        float* const tile = reinterpret_cast<float*>(lds);
        if (wn == 0) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        tot[r][t][v] = (tot[r][t][v] / (1.0f + expf(-tot[r][t][v]))) * ex[(((wm * 2 + r) * 2 + t) * 16 + v) * 64 + lane];
        }
        __syncthreads();
        if (wn == 0) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        tile[(wm * 64 + t * 32 + 8 * (v >> 2) + 4 * fo + (v & 3)) * 68 + r * 32 + (lane & 31)] = tot[r][t][v];
        }
        __syncthreads();
        if (a.yplanes) {
            const uint64_t plane = 2ull * a.yplanes * a.n;  // bytes of the high plane (n % 32 == 0)
            for (uint32_t i = tid; i < 128 * 8; i += 256) {
                const uint32_t t = i & 127, c8 = i >> 7, n = n0 + 8 * c8;
                if (t >= cnt || n >= a.n) continue;
                const uint64_t o = ((uint64_t)((n >> 5) * 4 + ((n >> 3) & 3)) * a.yplanes + t0 + t) * 16;
                bf16x8 hi, lo;
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float v = tile[t * 68 + 8 * c8 + k];
                    const __bf16 h = (__bf16)v;
                    hi[k] = h;
                    lo[k] = (__bf16)(v - (float)h);
                }
                gstore<bf16x8>(a.y + o, hi);
                gstore<bf16x8>(a.y + plane + o, lo);
            }
        } else {
            for (uint32_t i = tid; i < 128 * 64; i += 256) {
                const uint32_t t = i >> 6, n = n0 + (i & 63);
                if (t < cnt && n < a.n) gstore<float>(a.y + 4 * ((uint64_t)(t0 + t) * a.n + n), tile[t * 68 + (i & 63)]);
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const uint32_t n = n0 + wn * 64 + r * 32 + (lane & 31);
        if (n >= a.n) continue;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const uint32_t m = wm * 64 + t * 32 + 8 * (v >> 2) + 4 * fo + (v & 3);
                if (m >= cnt) continue;
                uint32_t yr = t0 + m;
                if (!dense) {
                    yr = jobs[m];
                    if (yr == QP_NOOFF) continue;
                }
                if (a.ws) {
                    gstore<float>(a.ws + 4 * (((uint64_t)split * a.rows + yr) * a.n + n), tot[r][t][v]);
                } else {
                    const uint64_t o = a.y + 4 * ((uint64_t)yr * a.n + n);
                    gstore<float>(o, a.acc ? gload<float>(o) + tot[r][t][v] : tot[r][t][v]);
                }
            }
    }
}

#define TILE_KERNELS(NAME, FMT)                                                                                       \
    KERNEL __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void qp_tile_##NAME(QpTileArgs a) {      \
        tile_body<FMT, false>(a);                                                                                     \
    }                                                                                                                 \
    KERNEL __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void qp_tile_glu_##NAME(QpTileArgs a) {  \
        tile_body<FMT, true>(a);                                                                                      \
    }
TILE_KERNELS(q4k, QP_Q4_K)
TILE_KERNELS(q5k, QP_Q5_K)
TILE_KERNELS(q6k, QP_Q6_K)
TILE_KERNELS(q3k, QP_Q3_K)
TILE_KERNELS(q2k, QP_Q2_K)
