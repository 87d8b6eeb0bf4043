// Dense int4 x fp16 products whose 128 x 256 tiles would leave most of the chip idle: the waves of a block share one small
// output tile and split its contraction between them.
#pragma once

#include "tf_prefill_kernels.hpp"

namespace tfk {

// Y[M, N] = X[M, K] . W[N, K]^T.  The tile kernels of tf_qmm.hip give a block 128 x 256 outputs and the whole of K: a block of 53 rows
// and 2048 columns makes 8 of them, each a chain of 44 dependent steps of about 0.65 us (28 us), and 120 rows of 2816 columns by
// 4096 make 11 (53 us).  Here a block owns 32 MT x 64 outputs and its NW waves take consecutive runs of K, so that the same product
// is 64 blocks of eight waves with six steps each.
//
// A wave is on its own until the end: its ring of three stages (32 MT activation rows x 64 k and 64 weight rows x 32 bytes each)
// is private, so there is no barrier in the loop; three stages are on their way while one is multiplied out of registers.  The scales
// and biases of the wave's rows over its run of K are fetched once, before the loop, one row a lane, and left in LDS as the fp16 pairs
// the expansion wants.  At the end the waves' fp32 sums meet in LDS and are added in wave order.
//
// RUNS: consecutive runs that K is cut into, one a wave, or RUNS / NW a wave one after the other: the same sums from fewer waves, for blocks that
// share a launch (and a compute unit) with the grouped tiles.
//
// A weight is half(q s + b), as in the tile kernels, with the same power of two for rows whose bf16 scales lie below fp16's normal
// range (a wave looks at all the scales of its run, so it never normalises less than the tile kernels do).
// GEGLU: the tile's two column tiles are 32 rows of the gate matrix and the same rows of the up matrix; the output is 32 columns
// of half(gelu_tanh(half(gate)) * half(up)).
struct SplitArgs {
    const uint8_t *W[2], *S[2], *B[2];
    const half_t *X;
    long ldx;
    half_t *Y;
    long ldy;
    int M, N, K;
    bool vec;                 // Y 8-byte aligned, N % 4 == 0, ldy % 4 == 0: four outputs a store
};

inline SplitArgs qmm_split_args(const uint8_t *w, const uint8_t *s, const uint8_t *b, const half_t *x, long ldx, half_t *y, long ldy, int m, int n, int k) {
    return SplitArgs{{w, w}, {s, s}, {b, b}, x, ldx, y, ldy, m, n, k, aligned(y, 8) && n % 4 == 0 && ldy % 4 == 0};
}
inline SplitArgs geglu_split_args(const tf_projection *gate, const tf_projection *up, const half_t *x, long ldx, half_t *a_out, long lda, int m) {
    const int f = (int)gate->rows, d = (int)gate->cols;
    return SplitArgs{{at(gate->weights, gate->weights_offset), at(up->weights, up->weights_offset)},
                     {at(gate->scales, gate->scales_offset), at(up->scales, up->scales_offset)},
                     {at(gate->biases, gate->biases_offset), at(up->biases, up->biases_offset)},
                     x, ldx, a_out, lda, m, f, d, aligned(a_out, 8) && f % 4 == 0 && lda % 4 == 0};
}

__device__ __forceinline__ void lds_write4(uint32_t addr, uint32_t v) { asm volatile("ds_write_b32 %0, %1" ::"v"(addr), "v"(v) : "memory"); }

// GP: most pairs of groups a run may have
template <int BITS, int MT, int NJ, int NW, int GP, int RUNS = NW>
struct SplitGeom {
    static constexpr int kWRow = 8 * BITS;                    // bytes of a weight row per step
    static constexpr int kWCopies = NJ * BITS / 4;
    static constexpr int kStage = MT * 4096 + NJ * 32 * kWRow;
    static constexpr int kCopies = MT * 4 + kWCopies;
    static constexpr int kSB = GP * 2 * 64 * 4;               // [group][row]: half(s) | half(b) << 16
    static constexpr int kWave = 3 * kStage + kSB;
    static constexpr int kSumRow = 32 * NJ + 4;                    // floats per row of a wave's sums
    static constexpr int kSums = 32 * MT * kSumRow * 4;       // one run's sums
    static constexpr int kLds = NW * kWave > RUNS * kSums ? NW * kWave : RUNS * kSums;
};

// One run of K for the tile at (m0, n0): acc += its products, post: what they are to be multiplied by, a power of two per column.  base:
// the wave's LDS; the wave leaves with nothing on its way into it and no read of it outstanding.
template <int BITS, int SD, int MT, int NJ, int NW, int GP, bool GEGLU, int RUNS>
__device__ __forceinline__ void qmm_split_run(const SplitArgs &a, int run, int m0, int n0, uint32_t base, int lane, float16_t (&acc)[MT][NJ], float (&post)[2]) {
    typedef SplitGeom<BITS, MT, NJ, NW, GP, RUNS> G;
    constexpr int kCols = GEGLU ? 32 : 32 * NJ;
    const int groups = a.K >> 6, pairs = (groups + 1) >> 1;
    const int g0 = 2 * (pairs * run / RUNS), g1 = min(groups, 2 * (pairs * (run + 1) / RUNS)), steps = g1 - g0;
    const uint32_t sb_area = base + 3 * G::kStage;
    const uint32_t row_bytes = (uint32_t)a.K * BITS / 8u;

    if (steps > 0) {
        // the lane's row of the tile as a copier of scales: row lane & 31 of column tile lane >> 5 (rows past the matrix: its last row)
        const int tile = lane >> 5, i = lane & 31, kb = lane >> 5;
        const int srow = min(n0 + (kCols == 32 ? i : lane), a.N - 1);
        const int which = GEGLU ? tile : 0;
        const uint8_t *sp = (which ? a.S[1] : a.S[0]) + ((size_t)srow * groups + g0) * 2, *bp = (which ? a.B[1] : a.B[0]) + ((size_t)srow * groups + g0) * 2;
        uint32_t sv[GP], bv[GP];
        const bool words = ((groups & 1) == 0) && ((((uintptr_t)a.S[0] | (uintptr_t)a.S[1] | (uintptr_t)a.B[0] | (uintptr_t)a.B[1]) & 3) == 0);
        // past the wave's run: its last values again (the copies of those groups are not read, and a maximum does not mind)
        if (words) {      // g0 is even: whole pairs
            const int last = (steps - 1) >> 1;
#pragma unroll
            for (int t = 0; t < GP; ++t) {
                sv[t] = reinterpret_cast<const uint32_t *>(sp)[min(t, last)];
                bv[t] = reinterpret_cast<const uint32_t *>(bp)[min(t, last)];
            }
        } else {
            const uint16_t *sh = reinterpret_cast<const uint16_t *>(sp), *bh = reinterpret_cast<const uint16_t *>(bp);
            uint16_t v[4 * GP];
#pragma unroll
            for (int t = 0; t < 2 * GP; ++t) {
                v[2 * t] = sh[min(t, steps - 1)];
                v[2 * t + 1] = bh[min(t, steps - 1)];
            }
#pragma unroll
            for (int t = 0; t < GP; ++t) {
                sv[t] = v[4 * t] | (uint32_t)v[4 * t + 2] << 16;
                bv[t] = v[4 * t + 1] | (uint32_t)v[4 * t + 3] << 16;
            }
        }
        // copies: activation rows 8 q + lane / 8, chunk (lane & 7) ^ ((row / 2) & 7); weight rows 32 q + lane / 2, 16-byte half
        // (lane & 1) ^ ((row / 4) & 1), or with 8 bits rows 16 q + lane / 4, piece (lane & 3) ^ ((row / 4) & 3).  Rows past the matrix repeat its last row; what they produce is not stored.
        qmm_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(a.X + (size_t)m0 * a.ldx), 0, (int)0xFFFFFFFFu, 0x00020000);
        qmm_rsrc_t wr[2];
        wr[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.W[0] + (size_t)n0 * row_bytes), 0, (int)0xFFFFFFFFu, 0x00020000);
        wr[1] = GEGLU ? __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.W[1] + (size_t)n0 * row_bytes), 0, (int)0xFFFFFFFFu, 0x00020000) : wr[0];
        uint32_t xoff[MT * 4], woff[G::kWCopies];
#pragma unroll
        for (int q = 0; q < MT * 4; ++q) {
            const int r = 8 * q + (lane >> 3);
            xoff[q] = (uint32_t)(min(m0 + r, a.M - 1) - m0) * (uint32_t)(a.ldx * 2) + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
        }
#pragma unroll
        for (int q = 0; q < G::kWCopies; ++q) {
            constexpr int kPieces = BITS / 2;      // 16-byte pieces of a row per step
            const int r = (64 / kPieces) * q + lane / kPieces;
            woff[q] = (uint32_t)(min(n0 + (GEGLU ? (r & 31) : r), a.N - 1) - n0) * row_bytes + (uint32_t)(((lane % kPieces) ^ ((r >> 2) % kPieces)) * 16);
        }
        auto copy = [&](int g, uint32_t stage) {
#pragma unroll
            for (int q = 0; q < G::kWCopies; ++q) lds_copy16(wr[q * NJ / G::kWCopies], stage + MT * 4096 + q * 1024, woff[q], g * G::kWRow);
#pragma unroll
            for (int q = 0; q < MT * 4; ++q) lds_copy16(xr, stage + q * 1024, xoff[q], g * 128);
        };
        copy(g0, base);
        if (steps > 1) copy(g0 + 1, base + G::kStage);
        if (steps > 2) copy(g0 + 2, base + 2 * G::kStage);

        uint32_t shift = 0;
        if constexpr (SD == 0) {
            // the power of two of the lane's row over the wave's run: every |s| < 2^(es - 126), every |b| < 2^(eb - 126), and
            // 2^(140 - max(es + BITS, eb)) brings q |s| + |b| below 2^15
            u16x2 es = {0, 0}, eb = {0, 0};
            bool small = false;
#pragma unroll
            for (int t = 0; t < GP; ++t) {
                es = __builtin_elementwise_max(es, __builtin_bit_cast(u16x2, sv[t] & 0x7F807F80u));
                eb = __builtin_elementwise_max(eb, __builtin_bit_cast(u16x2, bv[t] & 0x7F807F80u));
                const uint32_t lo = (sv[t] >> 7) & 0xFFu, hi = (sv[t] >> 23) & 0xFFu;
                small = small || (lo != 0u && lo < 113u) || (hi != 0u && hi < 113u);      // 2^-14 = fp16's smallest normal number
            }
            if (__builtin_amdgcn_ballot_w64(small) != 0ull) {
                const uint32_t top = max(((uint32_t)max(es[0], es[1]) >> 7) + (uint32_t)BITS, (uint32_t)max(eb[0], eb[1]) >> 7);
                const int e = top == (uint32_t)BITS ? 0 : min(max(140 - (int)top, -100), 100);
                shift = (uint32_t)e << 23;
                const float p = __uint_as_float((uint32_t)(127 - e) << 23);
                post[0] = __shfl(p, i, kWave);
                post[1] = __shfl(p, 32 + i, kWave);
            }
        }
#pragma unroll
        for (int t = 0; t < GP; ++t) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const half2_t s2 = sb_to_half2<SD>((uint16_t)(h ? sv[t] >> 16 : sv[t] & 0xFFFFu), shift);
                const half2_t b2 = sb_to_half2<SD>((uint16_t)(h ? bv[t] >> 16 : bv[t] & 0xFFFFu), shift);
                lds_write4(sb_area + (uint32_t)(2 * t + h) * 256u + (uint32_t)lane * 4u, as_u32(half2_t{s2[0], b2[0]}));
            }
        }

        struct Frags {
            u32x4 x[MT][4], w[NJ][BITS / 4];
            uint32_t sb[NJ];
        };
        const uint32_t x0 = (uint32_t)i * 128u + ((((uint32_t)kb * 4u) ^ (uint32_t)((i >> 1) & 7)) << 4);
        const uint32_t w0 = MT * 4096 + (uint32_t)i * (uint32_t)G::kWRow + (BITS == 4 ? (uint32_t)(kb ^ ((i >> 2) & 1)) << 4 : (uint32_t)((2 * kb) ^ ((i >> 2) & 3)) << 4);
        const uint32_t sb0 = sb_area + (uint32_t)i * 4u;
        auto read = [&](Frags &f, uint32_t stage, int t) {
            const uint32_t xa = stage + x0, wa = stage + w0, sa = sb0 + (uint32_t)t * 256u;
            f.w[0][0] = lds_read16<0>(wa);
            if constexpr (NJ > 1) f.w[NJ - 1][0] = lds_read16<32 * G::kWRow>(wa);
            if constexpr (BITS == 8) {                 // the other half of the lane's 32 bytes: the piece beside it
                f.w[0][BITS / 4 - 1] = lds_read16<0>(wa ^ 16u);
                if constexpr (NJ > 1) f.w[NJ - 1][BITS / 4 - 1] = lds_read16<32 * G::kWRow>(wa ^ 16u);
            }
            f.sb[0] = lds_read4<0>(sa);
            if constexpr (NJ > 1) f.sb[1] = lds_read4<128>(sa);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                f.x[0][d] = lds_read16<0>(xa ^ ((uint32_t)d << 4));
                if constexpr (MT > 1) f.x[1][d] = lds_read16<4096>(xa ^ ((uint32_t)d << 4));
            }
        };
        // all reads of f have landed; also keeps the copies that follow behind them
        auto landed = [&](Frags &f) {
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.w[0][0]), "+v"(f.sb[0]), "+v"(f.x[0][0]), "+v"(f.x[0][1]), "+v"(f.x[0][2]), "+v"(f.x[0][3]) : : "memory");
            if constexpr (NJ > 1) asm volatile("" : "+v"(f.w[NJ - 1][0]), "+v"(f.sb[NJ - 1]));
            if constexpr (BITS == 8) asm volatile("" : "+v"(f.w[0][BITS / 4 - 1]));
            if constexpr (BITS == 8 && NJ > 1) asm volatile("" : "+v"(f.w[NJ - 1][BITS / 4 - 1]));
            if constexpr (MT > 1) asm volatile("" : "+v"(f.x[1][0]), "+v"(f.x[1][1]), "+v"(f.x[1][2]), "+v"(f.x[1][3]));
        };
        uint32_t mask = 0x00F0000Fu;
        auto multiply = [&](const Frags &f) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                half8_t wf[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const half2_t sb = as_half2(f.sb[j]), s2 = {sb[0], sb[0]}, b2 = {sb[1], sb[1]};
                    const half2_t off = {(half_t)-1024.0f, (half_t)(BITS == 4 ? -64.0f : -1024.0f)};
                    u32x4 o;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        half2_t q;                                       // 1024 + q and 64 + q, or 1024 + q twice: exact
                        if constexpr (BITS == 4) {
                            const uint32_t both = __builtin_amdgcn_perm(0u, f.w[j][0][d], 0x0c000c00u | ((uint32_t)p << 16) | (uint32_t)p);
                            q = as_half2((both & mask) | 0x54006400u) + off;
                        } else {
                            q = as_half2(__builtin_amdgcn_perm(0x64646464u, f.w[j][(d >> 1) % (BITS / 4)][2 * (d & 1) + (p >> 1)], (p & 1) ? 0x04030402u : 0x04010400u)) + off;
                        }
                        o[p] = as_u32(__builtin_elementwise_fma(q, s2, b2));
                    }
                    wf[j] = __builtin_bit_cast(half8_t, o);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) acc[mt][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, f.x[mt][d]), wf[j], acc[mt][j], 0, 0, 0);
            }
        };
        // Step t: request stage t + 3 into the place stage t was read from, read stage t + 1 into registers, multiply stage t.
        // Requests still on their way when stage t + 1 must have landed: those of t + 2 and t + 3, as far as they exist.
        uint32_t cur = base;                       // where stage t lives
        auto wrap = [&](uint32_t s) { return s == base + 2 * G::kStage ? base : s + G::kStage; };
        auto arrive = [&](int younger) {
            if (younger >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * G::kCopies) : "memory");
            else if (younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(G::kCopies) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        };
        Frags f0, f1;
        arrive(min(steps - 1, 2));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the scales are in LDS (written and read by this wave only)
        read(f0, cur, 0);
        landed(f0);
        auto step = [&](int t, const Frags &now, Frags &next) {
            if (t + 3 < steps) copy(g0 + t + 3, cur);
            cur = wrap(cur);
            if (t + 1 < steps) {
                arrive(min(steps - t - 2, 2));
                read(next, cur, t + 1);
            }
            multiply(now);
            if (t + 1 < steps) landed(next);
        };
        for (int t = 0; t < steps; t += 2) {
            step(t, f0, f1);
            if (t + 1 < steps) step(t + 1, f1, f0);
        }
    }
}

// One tile of the product: 32 MT rows by 32 NJ columns (GEGLU: 32).  id: the block's number among those of the product, column tiles fastest
// and dealt to the XCDs in turn: the blocks of a row tile read the same activations, those of a column tile the same (four times smaller)
// weights; a block past the last tile does nothing.  lds: G::kLds bytes, 128-byte aligned.
template <int BITS, int SD, int MT, int NJ, int NW, int GP, bool GEGLU, int RUNS = NW>
__device__ __forceinline__ void qmm_split_body(const SplitArgs &a, uint32_t id, uint8_t *lds) {
    typedef SplitGeom<BITS, MT, NJ, NW, GP, RUNS> G;
    static_assert(!GEGLU || NJ == 2, "a gate tile and an up tile");
    static_assert(RUNS % NW == 0, "every wave takes the same number of runs");
    constexpr int kCols = GEGLU ? 32 : 32 * NJ, kRounds = RUNS / NW;
    const int lane = threadIdx.x & 63, wave = (int)uniform_u32(threadIdx.x >> 6);
    const int col_tiles = (a.N + kCols - 1) / kCols;
    const int n0 = (int)(id % (uint32_t)col_tiles) * kCols, m0 = (int)(id / (uint32_t)col_tiles) * 32 * MT;
    if (m0 >= a.M) return;
    const uint32_t base = (uint32_t)(uintptr_t)lds + (uint32_t)(wave * G::kWave);
    float16_t acc[kRounds][MT][NJ];
    float post[kRounds][2];
#pragma unroll
    for (int i = 0; i < kRounds; ++i) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][mt][j][r] = 0.0f;
        post[i][0] = post[i][1] = 1.0f;
        qmm_split_run<BITS, SD, MT, NJ, NW, GP, GEGLU, RUNS>(a, wave * kRounds + i, m0, n0, base, lane, acc[i], post[i]);
    }

    // the runs' sums -> LDS -> added in the order of the runs
    __syncthreads();
    float *const sums = reinterpret_cast<float *>(lds);
    constexpr int kRunFloats = G::kSums / 4;
#pragma unroll
    for (int i = 0; i < kRounds; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    sums[(wave * kRounds + i) * kRunFloats + (32 * mt + acc_row(r, lane)) * G::kSumRow + 32 * j + acc_col(lane)] = acc[i][mt][j][r] * post[i][j];
    __syncthreads();
    constexpr int kQuads = kCols / 4;              // pieces of four outputs in a row
    for (int idx = (int)threadIdx.x; idx < 32 * MT * kQuads; idx += 64 * NW) {
        const int row = idx / kQuads, col = (idx % kQuads) * 4;
        const int m = m0 + row, n = n0 + col;
        if (m >= a.M || n >= a.N) continue;
        auto total = [&](int c) {
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < RUNS; ++w) v += *reinterpret_cast<const f32x4 *>(sums + w * kRunFloats + row * G::kSumRow + c);
            return v;
        };
        f32x4 v = total(col);
        if constexpr (GEGLU) {
            const f32x4 up = total(32 + col);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (BITS == 4 ? gelu_tanh_fast((float)(half_t)v[e]) : gelu_tanh((float)(half_t)v[e])) * (float)(half_t)up[e];
        }
        half_t *y = a.Y + (size_t)m * a.ldy + n;
        if (a.vec) {
            *reinterpret_cast<half4_t *>(y) = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < a.N) y[e] = (half_t)v[e];
        }
    }
}

}  // namespace tfk
