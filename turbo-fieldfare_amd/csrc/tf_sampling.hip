// What sits either side of the tied int4 output head: the embedding row lookup (same table), the soft-capped softmax over
// the vocabulary, and the samplers (greedy, Gumbel-max, top-k / top-p / temperature with inverse-CDF draw).
// The reference runs each of these in a single threadgroup; here the vocabulary-sized passes are spread over the chip and
// meet through per-block partials (softmax), an atomic argmax fold (greedy, Gumbel) or the maxima of 64-element chunks (top-k).
#include "tf_argmax.hpp"
#include "tf_context.hpp"
#include "tf_rowdot.hpp"

using namespace tfk;

namespace {

// fp32 -> fp16 with the fp32 value pinned first, so that the multiply producing it is rounded to fp32 as in the
// reference and not fused into the conversion
__device__ __forceinline__ half_t to_half_pinned(float v) {
    asm volatile("" : "+v"(v));
    return (half_t)v;
}

// ------------------------------------------------------------------------------------------------ embedding rows
// out[t, i] = half((q * s + b) * out_scale) for row tokens[t] of the int4 table; one thread per 8 elements (one word).
__global__ __launch_bounds__(256) void embed_lookup_kernel(const uint8_t *table, const uint16_t *scales, const uint16_t *biases,
                                                           const uint32_t *tokens, uint32_t single_token, half_t *out, uint32_t rows,
                                                           uint32_t d, float out_scale, uint32_t table_rows) {
    const uint32_t t = blockIdx.y;
    const uint32_t word = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= rows || word * 8u >= d) return;
    uint32_t token = tokens ? tokens[t] : single_token;
    token = token < table_rows ? token : table_rows - 1;
    const uint32_t groups = d >> 6;
    const uint16_t *wp = reinterpret_cast<const uint16_t *>(table + (size_t)token * (d >> 1) + (size_t)word * 4);
    const uint32_t w = (uint32_t)wp[0] | ((uint32_t)wp[1] << 16);
    const float s = bf16_to_f32(scales[(size_t)token * groups + (word >> 3)]);
    const float b = bf16_to_f32(biases[(size_t)token * groups + (word >> 3)]);
    half_t *dst = out + (size_t)t * d + (size_t)word * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[i] = to_half_pinned(((float)((w >> (4 * i)) & 0xFu) * s + b) * out_scale);
}

// ------------------------------------------------------------------------------------------------ soft-capped softmax
// z = softcap * tanh(x / softcap); probs = exp(z - max z) / sum exp(z - max z).  First launch: per-block (max, sum) by
// the online rule; second launch: every block merges the partials (a few hundred values) and normalises its share.
constexpr uint32_t kSoftmaxMaxBlocks = 256;

__device__ __forceinline__ float softcapped(float x, float softcap) { return softcap * tanhf(x / softcap); }

// merge (m2, d2) into (m, d): d counts exp(z - m)
__device__ __forceinline__ void merge_md(float &m, float &d, float m2, float d2) {
    const float mn = fmaxf(m, m2);
    const float a = (m == -INFINITY) ? 0.0f : d * expf(m - mn);
    const float b = (m2 == -INFINITY) ? 0.0f : d2 * expf(m2 - mn);
    m = mn;
    d = a + b;
}

// reduces (m, d) over a 256-thread block; every thread gets the result.  scratch: 8 floats of LDS.
__device__ __forceinline__ void block_merge_md(float &m, float &d, float *scratch) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float m2 = __shfl_xor(m, off, kWave);
        const float d2 = __shfl_xor(d, off, kWave);
        merge_md(m, d, m2, d2);
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
        scratch[threadIdx.x >> 6] = m;
        scratch[4 + (threadIdx.x >> 6)] = d;
    }
    __syncthreads();
    m = scratch[0];
    d = scratch[4];
#pragma unroll
    for (int w = 1; w < 4; ++w) merge_md(m, d, scratch[w], scratch[4 + w]);
}

// Both launches are a chain of transcendental functions behind one load, not bandwidth (0.5 MB): a thread takes four neighbours
// (one load) and the online rule once per four, and a vocabulary of 262144 spreads over 256 blocks (softcap + softmax of 262144
// fp16 logits 4.6 us; 8.7 us with eight elements a thread taken one by one over 128 blocks).
constexpr uint32_t kSoftmaxRun = 4;

// logits [i, i + 4) below v; missing ones are -inf.  VEC: the row is aligned to whole runs
template <bool VEC, typename T>
__device__ __forceinline__ void load_run(const T *logits, uint32_t i, uint32_t v, float z[kSoftmaxRun]) {
    if (VEC && i < v && v - i >= kSoftmaxRun) {
        typedef T run_t __attribute__((ext_vector_type(kSoftmaxRun)));
        const run_t x = *reinterpret_cast<const run_t *>(logits + i);
#pragma unroll
        for (uint32_t j = 0; j < kSoftmaxRun; ++j) z[j] = (float)x[j];
    } else {
#pragma unroll
        for (uint32_t j = 0; j < kSoftmaxRun; ++j) z[j] = i < v && j < v - i ? (float)logits[i + j] : -INFINITY;
    }
}

template <bool VEC, typename T>
__global__ __launch_bounds__(256) void softmax_partials_kernel(const T *logits, float *partials, uint32_t v, float softcap) {
    __shared__ float scratch[8];
    float m = -INFINITY, d = 0.0f;
    // counted in runs: elements of a vocabulary near 2^32 would wrap and the loop never end
    for (uint32_t run = blockIdx.x * blockDim.x + threadIdx.x; run <= (v - 1) / kSoftmaxRun; run += gridDim.x * blockDim.x) {
        const uint32_t i = run * kSoftmaxRun;
        float z[kSoftmaxRun], mn = m;
        load_run<VEC>(logits, i, v, z);
#pragma unroll
        for (uint32_t j = 0; j < kSoftmaxRun; ++j) {
            z[j] = j < v - i ? softcapped(z[j], softcap) : -INFINITY;
            mn = fmaxf(mn, z[j]);
        }
        d = (m == -INFINITY) ? 0.0f : d * expf(m - mn);
#pragma unroll
        for (uint32_t j = 0; j < kSoftmaxRun; ++j)
            if (j < v - i) d += expf(z[j] - mn);
        m = mn;
    }
    block_merge_md(m, d, scratch);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = m;
        partials[2 * blockIdx.x + 1] = d;
    }
}

template <bool VEC, typename T>
__global__ __launch_bounds__(256) void softmax_normalize_kernel(const T *logits, const float *partials, uint32_t n_partials, half_t *probs,
                                                                uint32_t v, float softcap) {
    __shared__ float scratch[8];
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * kSoftmaxRun;
    float z[kSoftmaxRun];
    load_run<VEC>(logits, i, v, z);
    float m = -INFINITY, d = 0.0f;
    if (threadIdx.x < n_partials) {
        m = partials[2 * threadIdx.x];
        d = partials[2 * threadIdx.x + 1];
    }
#pragma unroll
    for (uint32_t j = 0; j < kSoftmaxRun; ++j) z[j] = softcapped(z[j], softcap);
    block_merge_md(m, d, scratch);
    const float inv_d = 1.0f / d;
    if (i >= v) return;
    half_t p[kSoftmaxRun];
#pragma unroll
    for (uint32_t j = 0; j < kSoftmaxRun; ++j) p[j] = to_half_pinned(expf(z[j] - m) * inv_d);
    if (VEC && v - i >= kSoftmaxRun) {
        typedef half_t run_t __attribute__((ext_vector_type(kSoftmaxRun)));
        *reinterpret_cast<run_t *>(probs + i) = run_t{p[0], p[1], p[2], p[3]};
    } else {
#pragma unroll
        for (uint32_t j = 0; j < kSoftmaxRun; ++j)
            if (j < v - i) probs[i + j] = p[j];
    }
}

template <typename T>
void launch_softmax(hipStream_t st, const T *logits, float *partials, half_t *probs, uint32_t v, float softcap) {
    const uint32_t runs = (v - 1) / (256 * kSoftmaxRun) + 1, blocks = runs < kSoftmaxMaxBlocks ? runs : kSoftmaxMaxBlocks;
    if (aligned16(logits) && aligned(probs, sizeof(half_t) * kSoftmaxRun)) {
        hipLaunchKernelGGL((softmax_partials_kernel<true, T>), dim3(blocks), dim3(256), 0, st, logits, partials, v, softcap);
        hipLaunchKernelGGL((softmax_normalize_kernel<true, T>), dim3(runs), dim3(256), 0, st, logits, partials, blocks, probs, v, softcap);
    } else {
        hipLaunchKernelGGL((softmax_partials_kernel<false, T>), dim3(blocks), dim3(256), 0, st, logits, partials, v, softcap);
        hipLaunchKernelGGL((softmax_normalize_kernel<false, T>), dim3(runs), dim3(256), 0, st, logits, partials, blocks, probs, v, softcap);
    }
}

// ------------------------------------------------------------------------------------------------ samplers
__device__ __forceinline__ uint64_t xorshift64(uint64_t &s) {
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return s * 2685821657736338717ull;
}
__device__ __forceinline__ float uniform01(uint64_t &s) { return (float)(uint32_t)(xorshift64(s) >> 40) * (1.0f / 16777216.0f); }

// counter-based Gumbel noise for (seed, position, row)
__device__ __forceinline__ float gumbel_for(uint64_t seed, uint32_t position, uint32_t row) {
    uint64_t x = seed ^ ((uint64_t)position * 0xD2B74407B1CE6E93ull) ^ (uint64_t)row;
    x = x + 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    x = x ^ (x >> 31);
    const float u = ((float)(uint32_t)(x >> 40) + 0.5f) * (1.0f / 16777216.0f);
    return -logf(-logf(u));
}

// GUMBEL false: argmax of the probabilities (temperature 0).  GUMBEL true: argmax of log(p) / T + Gumbel noise over the
// entries with p > 0, which draws from p^(1/T) / Z.  Ties go to the lowest index; nothing eligible gives token 0.
template <bool GUMBEL>
__global__ __launch_bounds__(256) void sample_argmax_kernel(const half_t *probs, uint32_t v, float inv_t, uint64_t seed, uint32_t position,
                                                            unsigned long long *cells, uint32_t *out_token) {
    __shared__ float sv[4];
    __shared__ uint32_t si[4];
    Best best{-INFINITY, 0xFFFFFFFFu};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < v; i += gridDim.x * blockDim.x) {
        const float p = (float)probs[i];
        if constexpr (GUMBEL) {
            if (!(p > 0.0f)) continue;
            const float s = inv_t * logf(p) + gumbel_for(seed, position, i);
            if (s > best.v) { best.v = s; best.idx = i; }
        } else {
            if (p > best.v) { best.v = p; best.idx = i; }
        }
    }
    wave_best_pair(best.v, best.idx);
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = best.v; si[threadIdx.x >> 6] = best.idx; }
    fold_block_best(sv, si, cells, out_token);
}

// ---- top-k
// The k best (k <= 256) of v probabilities by (value descending, index ascending) in two launches, without sorting the
// vocabulary.  fp16 values have 16-bit order-preserving keys, so "the k-th largest" is a binary search over at most 16
// thresholds, each a count of the elements that reach it (ballots and one block barrier):
//   1. chunk_max_kernel: the largest key of every 64 consecutive elements (one read of the probabilities by the whole chip);
//   2. topk_final_kernel, one block: T0 = the k-th largest of the chunk maxima.  At least k elements reach T0, so no element
//      below it is among the k best: only chunks whose maximum exceeds T0 (fewer than k) matter, and of those whose maximum is
//      T0 the first k (each holds an element equal to T0, and equal elements are taken by index).  The at most 2 k - 1 chunks
//      are read again (they are in the L2), their k-th largest key T1 is found the same way, ties at T1 are taken in index
//      order, and the k survivors are put in order by counting.
// Both launches are latency, not bandwidth (262144 probabilities are 0.5 MB); sorting every 1024-element tile with a bitonic
// network and merging the tiles in two more passes took 143 us at 262144, k = 64, where this takes 15.5 us, most of it the second launch.
// NaN and -inf are never chosen (key 0); -0 ties with 0.
constexpr uint32_t kTopkThreads = 1024, kTopkWaves = kTopkThreads / kWave;
constexpr uint32_t kTopkChunk = 64;
constexpr uint32_t kTopkCachedChunks = 4;                // chunk maxima a thread keeps in registers: 4096 of them, 262144 elements
constexpr uint32_t kTopkVocabFactor = 4;
constexpr uint32_t kTopkMaxK = 256;                      // the reference's working set (kSampleTopMaxK)

__device__ __forceinline__ uint32_t prob_key(uint16_t bits) {
    if (bits == 0x8000u) bits = 0u;
    const uint32_t key = (bits & 0x8000u) ? (uint32_t)(uint16_t)~bits : (uint32_t)bits | 0x8000u;
    const bool usable = (bits & 0x7FFFu) < 0x7C00u || bits == 0x7C00u;      // finite or +inf
    return usable ? key : 0u;
}
__device__ __forceinline__ float key_value(uint32_t key) {
    const uint16_t bits = (uint16_t)((key & 0x8000u) ? key & 0x7FFFu : ~key);
    return (float)__builtin_bit_cast(half_t, bits);
}

// VEC: probs is 16-byte aligned (a thread's eight elements in one load)
template <bool VEC>
__global__ __launch_bounds__(256) void chunk_max_kernel(const uint16_t *probs, uint16_t *chunk_max, uint32_t v) {
    const uint32_t piece = blockIdx.x * 256 + threadIdx.x, first = piece * 8;
    uint32_t best = 0;
    if (VEC && first < v && v - first >= 8) {
        const u32x4 w = *reinterpret_cast<const u32x4 *>(probs + first);
#pragma unroll
        for (int i = 0; i < 4; ++i) best = max(best, max(prob_key((uint16_t)w[i]), prob_key((uint16_t)(w[i] >> 16))));
    } else {
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i)
            if (first < v && i < v - first) best = max(best, prob_key(probs[first + i]));
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) best = max(best, (uint32_t)__shfl_xor((int)best, off, kWave));
    if ((threadIdx.x & 7) == 0 && first < v) chunk_max[piece >> 3] = (uint16_t)best;
}

// Sum of a wave-uniform count over the block's waves, in every thread.  `parity` alternates between two calls in a row, so one
// barrier a call is enough.
__device__ __forceinline__ uint32_t block_count(uint32_t wave_count, uint32_t (*cells)[kTopkWaves], uint32_t parity) {
    if ((threadIdx.x & 63) == 0) cells[parity][threadIdx.x >> 6] = wave_count;
    __syncthreads();
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t w = 0; w < kTopkWaves; ++w) sum += cells[parity][w];
    return sum;
}

// A threshold t in [lo, hi) that at least k keys of the block reach: the first one tried that at most `enough` reach, or else the
// largest (lo when fewer than k keys reach it).  count(t): how many of the wave's keys reach t; reached: how many of the
// block's reach the result (0 where that was never counted).
template <typename Count>
__device__ __forceinline__ uint32_t threshold(uint32_t lo, uint32_t hi, uint32_t k, uint32_t enough, uint32_t (*cells)[kTopkWaves], uint32_t &reached,
                                              Count count) {
    uint32_t parity = 0;
    reached = 0;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        const uint32_t n = block_count(count(mid), cells, parity);
        parity ^= 1;
        if (n >= k) {
            lo = mid;
            reached = n;
            if (n <= enough) break;
        } else {
            hi = mid;
        }
    }
    __syncthreads();      // the cells are free
    return lo;
}

__device__ __forceinline__ uint32_t lanes_before(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// table[0..N): exclusive running sum in place, by the first wave; the sum of all goes to *total.  Barriers before and after.
template <uint32_t N>
__device__ __forceinline__ void exclusive_scan(uint32_t *table, uint32_t *total) {
    static_assert(N % kWave == 0, "whole waves");
    __syncthreads();
    if (threadIdx.x < kWave) {
        uint32_t carry = 0;
#pragma unroll
        for (uint32_t i = threadIdx.x; i < N; i += kWave) {
            const uint32_t own = table[i];
            uint32_t sum = own;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const uint32_t up = (uint32_t)__shfl_up((int)sum, off, kWave);
                if ((int)threadIdx.x >= off) sum += up;
            }
            table[i] = carry + sum - own;
            carry += (uint32_t)__shfl((int)sum, kWave - 1, kWave);
        }
        if (threadIdx.x == 0) *total = carry;
    }
    __syncthreads();
}

// Running sums of `own` over a wave's lanes on top of `carry`, in lane order, one fp32 add per element: lane l holds what a
// sequential accumulation holds after element l, so a search over the lanes finds exactly the element a sequential walk would
// stop at.  A lane adds the elements up to its own and zeros from there on.
__device__ __forceinline__ float running_sums(float own, float carry) {
    float acc = carry;
#pragma unroll
    for (int j = 0; j < kWave; ++j) {
        const float x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(own), j));
        acc += (int)(threadIdx.x & 63) >= j ? x : 0.0f;
    }
    return acc;
}

// The sampler's tail, by one wave: slot 64 j + lane holds candidate number 64 j + lane, best first; only the first k slots (0 < k)
// count.  Follows the reference's sampler (Metal/Sampling/logit.metal:564-606): the usable prefix ends at the first slot that is
// empty or not finite; the top-p cut keeps the shortest prefix whose mass (probabilities still carry their full-vocabulary
// normalisation) reaches top_p; survivors are reweighted by p^(1/T); the draw is the inverse CDF of the seeded xorshift64* uniform.
// The sums that decide the cut and the draw are accumulated in index order.  Returns the chosen slot.
template <uint32_t SLOTS>
__device__ __forceinline__ uint32_t choose_slot(float value[SLOTS], const uint32_t index[SLOTS], uint32_t k, float temperature, float top_p,
                                                uint64_t seed) {
    const uint32_t lane = threadIdx.x & 63;
    auto first = [&](uint32_t none, auto holds) {      // lowest slot below `none` for which holds(j, slot)
        uint32_t found = none;
#pragma unroll
        for (uint32_t j = 0; j < SLOTS; ++j) {
            const uint64_t m = __ballot(64 * j + lane < none && holds(j));
            if (m != 0 && found == none) found = 64 * j + (uint32_t)__builtin_ctzll(m);
        }
        return found;
    };
    uint32_t n = first(k, [&](uint32_t j) { return index[j] == 0xFFFFFFFFu || !__builtin_isfinite(value[j]); });
    float sum[SLOTS];
    auto accumulate = [&]() {      // returns the sum of the first n
        float carry = 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < SLOTS; ++j) {
            sum[j] = carry;
            if (64 * j < n) {
                sum[j] = running_sums(64 * j + lane < n ? value[j] : 0.0f, carry);
                carry = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sum[j]), kWave - 1));
            }
        }
        return carry;
    };
    if (top_p > 0.0f && top_p < 1.0f) {
        (void)accumulate();
        const uint32_t last = first(n, [&](uint32_t j) { return sum[j] >= top_p; });
        n = last < n ? last + 1 : n;
    }
    if (temperature != 1.0f) {
#pragma unroll
        for (uint32_t j = 0; j < SLOTS; ++j)
            if (64 * j + lane < n) value[j] = powf(value[j], 1.0f / temperature);
    }
    const float mass = accumulate();
    uint64_t rng = seed;
    (void)xorshift64(rng);
    const float u = uniform01(rng) * mass;
    const uint32_t slot = first(n, [&](uint32_t j) { return u <= sum[j]; });
    return slot < n ? slot : 0;
}

// One block.  EPT: elements a thread looks after (EPT * 1024 >= (2 k - 1) * 64, or >= v where every element is looked at and
// chunk_max is null).
template <uint32_t EPT>
__global__ __launch_bounds__(kTopkThreads) void topk_final_kernel(const uint16_t *probs, const uint16_t *chunk_max, uint32_t v, uint32_t k,
                                                                  float temperature, float top_p, uint64_t seed, uint32_t *out_token) {
    constexpr uint32_t kMaxK = EPT <= 8 ? 64 : kTopkMaxK, kRounds = kTopkCachedChunks;
    constexpr uint32_t kChunkCapacity = EPT * kTopkThreads / kTopkChunk;      // 128 / 512: at least 2 k
    __shared__ uint32_t cells[2][kTopkWaves];
    __shared__ uint32_t table[EPT * kTopkWaves], taken_table[kRounds * kTopkWaves];
    __shared__ uint32_t chunk_list[kChunkCapacity];
    __shared__ uint64_t best[kMaxK];
    __shared__ uint32_t ranks[kMaxK];
    __shared__ float values[kMaxK];
    __shared__ uint32_t indices[kMaxK];
    __shared__ uint32_t word, total;
    const uint32_t t = threadIdx.x, wave = t >> 6;
    uint32_t listed = 0, floor_key = 1;      // chunks to look into; a key that at least k elements reach, if k are usable
    if (t == 0) total = 0;
    if (t < kMaxK) {
        ranks[t] = 0;
        values[t] = -INFINITY;
        indices[t] = 0xFFFFFFFFu;
        best[t] = 0;
    }
    if (chunk_max) {
        const uint32_t chunks = (v - 1) / kTopkChunk + 1, rounds = (chunks + kTopkThreads - 1) / kTopkThreads;
        auto maximum = [&](uint32_t r) { return r * kTopkThreads + t < chunks ? (uint32_t)chunk_max[r * kTopkThreads + t] : 0u; };
        uint32_t cached[kRounds];
#pragma unroll
        for (uint32_t r = 0; r < kRounds; ++r) cached[r] = maximum(r);
        uint32_t reached;
        const uint32_t t0 = threshold(1, 0x10000u, k, kChunkCapacity, cells, reached, [&](uint32_t mid) {
            uint32_t n = 0;
#pragma unroll
            for (uint32_t r = 0; r < kRounds; ++r) n += (uint32_t)__popcll(__ballot(cached[r] >= mid));
            for (uint32_t r = kRounds; r < rounds; ++r) n += (uint32_t)__popcll(__ballot(maximum(r) >= mid));
            return n;
        });
        floor_key = t0;
        const bool few = reached <= kChunkCapacity;      // every chunk that reaches T0 fits the list
        // the chosen chunks in index order: those that reach T0, or all above T0 and the first k at T0
        uint32_t ties = 0;
        for (uint32_t r0 = 0; r0 < rounds; r0 += kRounds) {
            uint32_t m[kRounds];
            bool take[kRounds];
#pragma unroll
            for (uint32_t r = 0; r < kRounds; ++r) {
                m[r] = r0 == 0 ? cached[r] : maximum(r0 + r);
                take[r] = m[r] >= t0;
            }
            if (!few) {
#pragma unroll
                for (uint32_t r = 0; r < kRounds; ++r) {
                    const uint64_t eq = __ballot(m[r] == t0);
                    if ((t & 63) == 0) taken_table[r * kTopkWaves + wave] = (uint32_t)__popcll(eq);
                }
                exclusive_scan<kRounds * kTopkWaves>(taken_table, &word);
#pragma unroll
                for (uint32_t r = 0; r < kRounds; ++r) {
                    const uint64_t eq = __ballot(m[r] == t0);
                    take[r] = m[r] > t0 || (m[r] == t0 && ties + taken_table[r * kTopkWaves + wave] + lanes_before(eq) < k);
                }
                ties += word;
                __syncthreads();
            }
#pragma unroll
            for (uint32_t r = 0; r < kRounds; ++r) {
                const uint64_t mask = __ballot(take[r]);
                if ((t & 63) == 0) taken_table[r * kTopkWaves + wave] = (uint32_t)__popcll(mask);
            }
            exclusive_scan<kRounds * kTopkWaves>(taken_table, &word);
#pragma unroll
            for (uint32_t r = 0; r < kRounds; ++r) {
                const uint64_t mask = __ballot(take[r]);
                if (take[r]) chunk_list[listed + taken_table[r * kTopkWaves + wave] + lanes_before(mask)] = (r0 + r) * kTopkThreads + t;
            }
            listed += word;
            __syncthreads();
        }
    }
    auto element = [&](uint32_t j) {      // slot j of this thread -> index in probs; slots ascend by index
        const uint32_t slot = j * kTopkThreads + t;
        if (!chunk_max) return slot;
        return slot / kTopkChunk < listed ? chunk_list[slot / kTopkChunk] * kTopkChunk + slot % kTopkChunk : v;
    };
    uint32_t key[EPT];
#pragma unroll
    for (uint32_t j = 0; j < EPT; ++j) {
        const uint32_t i = element(j);
        key[j] = i < v ? (uint32_t)probs[i] : 0xFFFFu;
    }
#pragma unroll
    for (uint32_t j = 0; j < EPT; ++j) key[j] = prob_key((uint16_t)key[j]);      // 0xFFFF is a NaN: never chosen
    uint32_t reached;
    const uint32_t t1 = threshold(floor_key, 0x10000u, k, k, cells, reached, [&](uint32_t mid) {
        uint32_t n = 0;
#pragma unroll
        for (uint32_t j = 0; j < EPT; ++j) n += (uint32_t)__popcll(__ballot(key[j] >= mid));
        return n;
    });
    // exactly the keys that reach T1 where k of them do; otherwise everything above T1 and the first of those at T1: `table` counts
    // the ties of every (j, wave), in index order
    uint32_t ties_wanted = 0xFFFFFFFFu;
    if (reached != k) {
        uint32_t above = 0;
#pragma unroll
        for (uint32_t j = 0; j < EPT; ++j) {
            const uint64_t eq = __ballot(key[j] == t1);
            above += (uint32_t)__popcll(__ballot(key[j] > t1));
            if ((t & 63) == 0) table[j * kTopkWaves + wave] = (uint32_t)__popcll(eq);
        }
        ties_wanted = k - block_count(above, cells, 0);
        exclusive_scan<EPT * kTopkWaves>(table, &word);
    }
#pragma unroll
    for (uint32_t j = 0; j < EPT; ++j) {
        bool take = key[j] >= t1;
        if (reached != k) {
            const uint64_t eq = __ballot(key[j] == t1);
            take = key[j] > t1 || (key[j] == t1 && table[j * kTopkWaves + wave] + lanes_before(eq) < ties_wanted);
        }
        if (take) best[atomicAdd(&total, 1u)] = ((uint64_t)key[j] << 32) | (uint64_t)(0xFFFFFFFFu - element(j));
    }
    __syncthreads();
    // a candidate's place is the number of better ones: candidate t % kMaxK against a share of the list (empty places hold 0)
    {
        constexpr uint32_t kShares = kTopkThreads / kMaxK, kShare = kMaxK / kShares;
        const uint64_t own = best[t % kMaxK];
        uint32_t better = 0;
#pragma unroll 4
        for (uint32_t j = 0; j < kShare; ++j) better += best[(t / kMaxK) * kShare + j] > own ? 1u : 0u;
        if (better) atomicAdd(&ranks[t % kMaxK], better);
    }
    __syncthreads();
    if (t < total) {
        values[ranks[t]] = key_value((uint32_t)(best[t] >> 32));
        indices[ranks[t]] = 0xFFFFFFFFu - (uint32_t)best[t];
    }
    __syncthreads();
    if (t < kWave) {
        constexpr uint32_t kSlots = kMaxK / kWave;
        float value[kSlots];
        uint32_t index[kSlots];
#pragma unroll
        for (uint32_t j = 0; j < kSlots; ++j) {
            value[j] = values[64 * j + t];
            index[j] = indices[64 * j + t];
        }
        const uint32_t slot = choose_slot<kSlots>(value, index, k, temperature, top_p, seed);
        if (t == 0) {
            const uint32_t token = indices[slot];
            out_token[0] = token == 0xFFFFFFFFu ? 0u : token;
        }
    }
}

// Wrapper-owned scratch of the samplers: [argmax cells + ticket | softmax partials | chunk maxima].
struct SampleScratch {
    unsigned long long *cells;
    float *partials;
    uint16_t *chunk_max;
};

constexpr size_t kCellBytes = (kHeadCells + 1) * sizeof(unsigned long long);
constexpr size_t kPartialBytes = kSoftmaxMaxBlocks * 2 * sizeof(float);

size_t sample_need(size_t elements) { return kCellBytes + kPartialBytes + (elements / kTopkChunk + 1) * sizeof(uint16_t); }

// The truncating samplers take vocabularies up to the limit in whole 1024 elements, four times as many for k <= 64
size_t topk_admitted(uint32_t max_vocab) { return ((size_t)max_vocab + 1023) / 1024 * 1024; }

int32_t sample_scratch(tf_ctx *ctx, size_t elements, SampleScratch &out) {
    const size_t need = sample_need(elements);
    if (ctx->sample_scratch_bytes < need) return scratch_too_small(ctx, "sampler", need, ctx->sample_scratch_bytes);
    uint8_t *base = static_cast<uint8_t *>(ctx->sample_scratch);
    out.cells = reinterpret_cast<unsigned long long *>(base);
    out.partials = reinterpret_cast<float *>(base + kCellBytes);
    out.chunk_max = reinterpret_cast<uint16_t *>(base + kCellBytes + kPartialBytes);
    return TF_OK;
}

uint32_t spread_blocks(const tf_ctx *ctx, uint32_t v, uint32_t cap) {
    const uint32_t by_work = (v + 2047) / 2048;             // at least 8 elements per thread
    uint32_t blocks = by_work < cap ? by_work : cap;
    const uint32_t chip = (uint32_t)ctx->num_cus * 2;
    blocks = blocks < chip ? blocks : chip;
    return blocks > 0 ? blocks : 1;
}

// the k best of probs[0..v) -> one token; k <= 256.  A vocabulary that one block can hold in registers takes the second launch
// alone.
int32_t launch_truncating_sampler(tf_ctx *ctx, hipStream_t st, const half_t *probs, uint32_t v, uint32_t k, float temperature, float top_p,
                                  uint64_t seed, uint32_t *out_token, const char *who) {
    const uint16_t *bits = reinterpret_cast<const uint16_t *>(probs);
    const uint32_t most = (k <= 64 ? 8u : 32u) * kTopkThreads;      // elements the final block looks at: (2 k - 1) chunks fit
    uint16_t *chunk_max = nullptr;
    if (v > most) {
        SampleScratch sc;
        const size_t admitted = topk_admitted(ctx->limits.max_vocab) * (k <= 64 ? kTopkVocabFactor : 1u);
        if (v > admitted) return scratch_too_small(ctx, "sampler", sample_need(v), sample_need(admitted));
        const int32_t rc = sample_scratch(ctx, v, sc);
        if (rc != TF_OK) return rc;
        chunk_max = sc.chunk_max;
        const dim3 grid((v - 1) / 2048 + 1);
        if (aligned16(probs)) hipLaunchKernelGGL(chunk_max_kernel<true>, grid, dim3(256), 0, st, bits, chunk_max, v);
        else hipLaunchKernelGGL(chunk_max_kernel<false>, grid, dim3(256), 0, st, bits, chunk_max, v);
    }
    if (k <= 64) hipLaunchKernelGGL(topk_final_kernel<8>, dim3(1), dim3(kTopkThreads), 0, st, bits, chunk_max, v, k, temperature, top_p, seed, out_token);
    else hipLaunchKernelGGL(topk_final_kernel<32>, dim3(1), dim3(kTopkThreads), 0, st, bits, chunk_max, v, k, temperature, top_p, seed, out_token);
    return check_launch(ctx, who);
}

}  // namespace

namespace tfk {

size_t sample_scratch_bytes_for(uint32_t vocab) { return sample_need(kTopkVocabFactor * topk_admitted(vocab)); }
size_t sample_scratch_clear_bytes() { return kCellBytes; }

}  // namespace tfk

extern "C" {

int32_t tf_embed_lookup_int4(tf_ctx *ctx, tf_stream stream, const void *table, uint64_t table_offset, const void *scales,
                             uint64_t scales_offset, const void *biases, uint64_t biases_offset, void *out, uint64_t out_offset,
                             uint32_t token_id, uint32_t d, float out_scale, uint32_t table_rows) {
    TF_REQUIRE(ctx, ctx && table && scales && biases && out, TF_ERR_INVALID_ARGUMENT, "embed_lookup_int4: null argument");
    TF_REQUIRE(ctx, d > 0 && d % TF_GROUP_SIZE == 0, TF_ERR_INVALID_ARGUMENT, "embed_lookup_int4: D must be a multiple of 64, got %u", d);
    TF_REQUIRE(ctx, token_id < table_rows, TF_ERR_INVALID_ARGUMENT, "embed_lookup_int4: token %u out of range (%u rows)", token_id, table_rows);
    const uint8_t *tb = at(table, table_offset);
    const uint8_t *sc = at(scales, scales_offset);
    const uint8_t *bi = at(biases, biases_offset);
    uint8_t *o = at(out, out_offset);
    TF_REQUIRE(ctx, aligned(tb, 2) && aligned(sc, 2) && aligned(bi, 2) && aligned(o, 2), TF_ERR_INVALID_ARGUMENT, "embed_lookup_int4: misaligned operand");
    hipLaunchKernelGGL(embed_lookup_kernel, dim3((d / 8 + 255) / 256, 1), dim3(256), 0, static_cast<hipStream_t>(stream), tb,
                       reinterpret_cast<const uint16_t *>(sc), reinterpret_cast<const uint16_t *>(bi), (const uint32_t *)nullptr, token_id,
                       reinterpret_cast<half_t *>(o), 1u, d, out_scale, table_rows);
    return check_launch(ctx, "embed_lookup_int4");
}

int32_t tf_prefill_embed_lookup_int4_block(tf_ctx *ctx, tf_stream stream, const void *table, uint64_t table_offset, const void *scales,
                                           uint64_t scales_offset, const void *biases, uint64_t biases_offset, const void *tokens,
                                           uint64_t tokens_offset, void *out, uint64_t out_offset, uint32_t t, uint32_t d, float out_scale,
                                           uint32_t table_rows) {
    TF_REQUIRE(ctx, ctx && table && scales && biases && tokens && out, TF_ERR_INVALID_ARGUMENT, "prefill_embed_lookup_int4_block: null argument");
    TF_REQUIRE(ctx, d > 0 && d % TF_GROUP_SIZE == 0, TF_ERR_INVALID_ARGUMENT, "prefill_embed_lookup_int4_block: D must be a multiple of 64, got %u", d);
    TF_REQUIRE(ctx, t > 0 && t <= 65535 && table_rows > 0, TF_ERR_INVALID_ARGUMENT, "prefill_embed_lookup_int4_block: t must be in 1...65535 and the table non-empty");
    const uint8_t *tb = at(table, table_offset);
    const uint8_t *sc = at(scales, scales_offset);
    const uint8_t *bi = at(biases, biases_offset);
    const uint8_t *tk = at(tokens, tokens_offset);
    uint8_t *o = at(out, out_offset);
    TF_REQUIRE(ctx, aligned(tb, 2) && aligned(sc, 2) && aligned(bi, 2) && aligned(o, 2) && aligned(tk, 4), TF_ERR_INVALID_ARGUMENT,
               "prefill_embed_lookup_int4_block: misaligned operand");
    hipLaunchKernelGGL(embed_lookup_kernel, dim3((d / 8 + 255) / 256, t), dim3(256), 0, static_cast<hipStream_t>(stream), tb,
                       reinterpret_cast<const uint16_t *>(sc), reinterpret_cast<const uint16_t *>(bi), reinterpret_cast<const uint32_t *>(tk), 0u,
                       reinterpret_cast<half_t *>(o), t, d, out_scale, table_rows);
    return check_launch(ctx, "prefill_embed_lookup_int4_block");
}

int32_t tf_logit_softcap_softmax(tf_ctx *ctx, tf_stream stream, const void *logits, void *probs, uint32_t v, float softcap,
                                 tf_dtype logits_dtype) {
    TF_REQUIRE(ctx, ctx && logits && probs, TF_ERR_INVALID_ARGUMENT, "logit_softcap_softmax: null argument");
    TF_REQUIRE(ctx, v > 0, TF_ERR_INVALID_ARGUMENT, "logit_softcap_softmax: V must be positive");
    TF_REQUIRE(ctx, softcap > 0.0f, TF_ERR_INVALID_ARGUMENT, "logit_softcap_softmax: softcap must be positive");
    TF_REQUIRE(ctx, logits_dtype == TF_FP16 || logits_dtype == TF_FP32, TF_ERR_INVALID_ARGUMENT, "logit_softcap_softmax: logits must be fp16 or fp32");
    TF_REQUIRE(ctx, aligned(logits, logits_dtype == TF_FP16 ? 2 : 4) && aligned(probs, 2), TF_ERR_INVALID_ARGUMENT, "logit_softcap_softmax: misaligned operand");
    SampleScratch sc;
    const int32_t rc = sample_scratch(ctx, 0, sc);
    if (rc != TF_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    half_t *ph = static_cast<half_t *>(probs);
    if (logits_dtype == TF_FP16) launch_softmax(st, static_cast<const half_t *>(logits), sc.partials, ph, v, softcap);
    else launch_softmax(st, static_cast<const float *>(logits), sc.partials, ph, v, softcap);
    return check_launch(ctx, "logit_softcap_softmax");
}

int32_t tf_sample(tf_ctx *ctx, tf_stream stream, const void *probs, void *out_token, uint32_t v, float temperature, uint32_t top_k,
                  float top_p, uint64_t seed, uint32_t position) {
    TF_REQUIRE(ctx, ctx && probs && out_token, TF_ERR_INVALID_ARGUMENT, "sample: null argument");
    TF_REQUIRE(ctx, v > 0, TF_ERR_INVALID_ARGUMENT, "sample: V must be positive");
    TF_REQUIRE(ctx, aligned(probs, 2) && aligned(out_token, 4), TF_ERR_INVALID_ARGUMENT, "sample: misaligned operand");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const half_t *ph = static_cast<const half_t *>(probs);
    uint32_t *tok = static_cast<uint32_t *>(out_token);
    const bool greedy = temperature <= 0.0f;
    if (greedy || (top_k == 0u && (top_p <= 0.0f || top_p >= 1.0f))) {
        SampleScratch sc;
        const int32_t rc = sample_scratch(ctx, 0, sc);
        if (rc != TF_OK) return rc;
        const uint32_t blocks = spread_blocks(ctx, v, 1024);
        if (greedy) hipLaunchKernelGGL(sample_argmax_kernel<false>, dim3(blocks), dim3(256), 0, st, ph, v, 0.0f, seed, position, sc.cells, tok);
        else hipLaunchKernelGGL(sample_argmax_kernel<true>, dim3(blocks), dim3(256), 0, st, ph, v, 1.0f / temperature, seed, position, sc.cells, tok);
        return check_launch(ctx, "sample");
    }
    uint32_t k = top_k == 0u ? v : top_k;
    k = k < 256u ? k : 256u;       // the reference's working set (kSampleTopMaxK)
    k = k < v ? k : v;
    return launch_truncating_sampler(ctx, st, ph, v, k, temperature, top_p, seed, tok, "sample");
}

int32_t tf_sample_topk64(tf_ctx *ctx, tf_stream stream, const void *probs, void *out_token, uint32_t vocab, float temperature, float top_p,
                         uint64_t seed) {
    TF_REQUIRE(ctx, ctx && probs && out_token, TF_ERR_INVALID_ARGUMENT, "sample_topk64: null argument");
    TF_REQUIRE(ctx, vocab > 0 && vocab <= 262144, TF_ERR_INVALID_ARGUMENT, "sample_topk64: unsupported vocabulary %u", vocab);
    TF_REQUIRE(ctx, temperature > 0.0f, TF_ERR_INVALID_ARGUMENT, "sample_topk64: temperature must be positive (greedy decoding takes the argmax path)");
    TF_REQUIRE(ctx, aligned(probs, 2) && aligned(out_token, 4), TF_ERR_INVALID_ARGUMENT, "sample_topk64: misaligned operand");
    return launch_truncating_sampler(ctx, static_cast<hipStream_t>(stream), static_cast<const half_t *>(probs), vocab, 64u < vocab ? 64u : vocab,
                                     temperature, top_p, seed, static_cast<uint32_t *>(out_token), "sample_topk64");
}

}  // extern "C"
