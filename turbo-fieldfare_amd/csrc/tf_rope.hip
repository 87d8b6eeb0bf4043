// Rotary position embedding (NeoX pairing) and the per-head Q/K/V epilogue: RMSNorm per head (q and k with a bf16 weight
// shared by all heads, v without), then rotation of the first `rotated_pairs` pairs of q and k, in place.  For one token
// (decode) and for a block of tokens at consecutive positions with padded token rows (prefill): the same kernels, so a block
// equals its tokens done one by one, bit for bit.
#include <math.h>

#include <type_traits>

#include "tf_common.hpp"
#include "tf_context.hpp"
#include "tf_epilogue_heads.hpp"

using namespace tfk;

namespace {

constexpr uint32_t kEpilogueBlocks = 2048;       // eight blocks of four waves a CU
constexpr uint32_t kEpilogueMaxHeadDim = 512;   // the reference's threadgroup scratch (fused.metal kFusedMaxHeadDim)

// (x0, x1) rotated by angle position * theta^(-2 pair / head_dim); accurate sine / cosine: angles reach position itself
__device__ __forceinline__ float rope_frequency(uint32_t pair, uint32_t head_dim, float theta) {
    return powf(theta, -(float)(2u * pair) / (float)head_dim);
}
__device__ __forceinline__ void rotate(float &x0, float &x1, float sn, float c) {
    const float r0 = x0 * c - x1 * sn, r1 = x0 * sn + x1 * c;
    x0 = r0;
    x1 = r1;
}
__device__ __forceinline__ void rope_pair(float &x0, float &x1, uint32_t pair, uint32_t head_dim, float position, float theta) {
    float sn, c;
    sincosf(position * rope_frequency(pair, head_dim, theta), &sn, &c);
    rotate(x0, x1, sn, c);
}

// grid (pair blocks, heads, tokens): head h of token t starts at t * token_stride + h * head_dim and sits at position
// position + t * position_step
__global__ __launch_bounds__(256) void rope_neox_kernel(half_t *data, uint32_t position, uint32_t position_step, uint32_t head_dim,
                                                        uint32_t token_stride, float theta, uint32_t rotated_pairs) {
    const uint32_t pair = blockIdx.x * blockDim.x + threadIdx.x;
    if (pair >= rotated_pairs) return;
    const uint32_t half_dim = head_dim / 2;
    half_t *head = data + (size_t)blockIdx.z * token_stride + (size_t)blockIdx.y * head_dim;
    float x0 = (float)head[pair], x1 = (float)head[half_dim + pair];
    rope_pair(x0, x1, pair, head_dim, (float)(position + blockIdx.z * position_step), theta);
    head[pair] = (half_t)x0;
    head[half_dim + pair] = (half_t)x1;
}

// Heads of 64 / 128 / 256 / 512: a wave per head, EPL = head_dim / 64 neighbouring elements a lane, all in registers; the partner
// of an element (NeoX pairing, head_dim / 2 away) sits 32 lanes further.  What bounds the step is the rotation angle - powf and
// sincosf, some 200 instructions - not the bytes, and the angle depends on (token, pair) only: the block computes the token's
// sines and cosines once, into LDS, for all of its heads (four at a time, heads_per_wave rounds).  With a block per head and an
// angle per head the step took 91 us at 2048 tokens x 32 heads of 256 (33.5 MB read and written).
// With eight heads a wave all waves of a call are resident at once and what is left is the issue of vector instructions, a hundred and eighty
// a head: angles and weights read again for every head, partners fetched through LDS, a square root and a division in all lanes for one
// number.  So a wave asks for all of its heads at the start, keeps both weights and its lanes' angles in registers, gets (x0, x1) from one
// lane swap, and takes the square roots and divisions of all heads in one go, head r's in lane r.
// 82 instructions a head.  2048 tokens x 32 heads of 256: 21.0 -> 15.6 us; 500 tokens: 10.1 -> 9.1; one token 3.4 -> 2.9; 20 heads of 512, 128
// tokens: 5.4 -> 4.5 (kernel times under the profiler).
// grid (head groups, tokens).  VEC: every head starts at a multiple of its lanes' piece (16 bytes at most).  HPW: heads a wave.  The arithmetic
// does not depend on VEC or HPW: a block of tokens equals its tokens done one by one, bit for bit.
template <int EPL, bool VEC, int HPW>
__global__ __launch_bounds__(256) void qkv_epilogue_wave_kernel(half_t *q, half_t *k, half_t *v, const uint16_t *q_weight, const uint16_t *k_weight,
                                                                uint32_t num_q_heads, uint32_t num_kv_heads, uint32_t position, float theta,
                                                                uint32_t rotated_pairs, float eps, uint32_t q_token_stride, uint32_t kv_token_stride) {
    constexpr uint32_t kHeadDim = EPL * 64, kHalfDim = kHeadDim / 2;
    typedef half_t piece_t __attribute__((ext_vector_type(EPL)));
    __shared__ float cosine[kHalfDim], sine[kHalfDim];
    const uint32_t t = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const EpilogueHeads kinds = {num_q_heads, num_kv_heads};
    const uint32_t heads = kinds.count(), head0 = blockIdx.x * 4 * HPW + wave;
    auto head_at = [&](uint32_t h) {
        return h < num_q_heads ? q + (size_t)t * q_token_stride + (size_t)h * kHeadDim
               : h < num_q_heads + num_kv_heads ? k + (size_t)t * kv_token_stride + (size_t)(h - num_q_heads) * kHeadDim
                                                : v + (size_t)t * kv_token_stride + (size_t)(h - num_q_heads - num_kv_heads) * kHeadDim;
    };
    piece_t piece[HPW];
#pragma unroll
    for (int r = 0; r < HPW; ++r) {
        const half_t *src = head_at(kinds.read(head0 + 4 * r)) + lane * EPL;
        if constexpr (VEC) {
            piece[r] = *reinterpret_cast<const piece_t *>(src);
        } else {
#pragma unroll
            for (int j = 0; j < EPL; ++j) piece[r][j] = src[j];
        }
    }
    // the weights of the wave's first and of its last head: q heads come first, so there are no others
    float first_w[EPL], last_w[EPL];
    const bool first_q = kinds.takes_q_weight(head0), last_q = kinds.takes_q_weight(head0 + 4 * (HPW - 1));
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        first_w[j] = bf16_to_f32((first_q ? q_weight : k_weight)[lane * EPL + j]);
        last_w[j] = HPW > 1 ? bf16_to_f32((last_q ? q_weight : k_weight)[lane * EPL + j]) : first_w[j];
    }
    for (uint32_t pair = threadIdx.x; pair < rotated_pairs; pair += blockDim.x) {
        float sn, c;
        sincosf((float)(position + t) * rope_frequency(pair, kHeadDim, theta), &sn, &c);
        cosine[pair] = c;
        sine[pair] = sn;
    }
    // 1 / rms of head r
    auto inverse = [&](float sum) { return 1.0f / sqrtf(sum / (float)kHeadDim + eps); };
    float sums = 0.0f;
#pragma unroll
    for (int r = 0; r < HPW; ++r) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < EPL; ++j) acc = fmaf((float)piece[r][j], (float)piece[r][j], acc);
        acc = wave_sum(acc);
        sums = HPW == 1 ? acc : (int)lane == r ? acc : sums;
    }
    const float invs = inverse(sums);
    __syncthreads();
    // element j of a lane: x0 of its pair times x0_by[j] plus x1 times x1_by[j]
    const bool is_x0 = lane < 32;
    float x0_by[EPL], x1_by[EPL];
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const uint32_t pair = (lane & 31) * EPL + j;
        const float sn = sine[pair], c = cosine[pair];      // beyond rotated_pairs: never used
        x0_by[j] = is_x0 ? c : sn;
        x1_by[j] = is_x0 ? -sn : c;
    }
#pragma unroll
    for (int r = 0; r < HPW; ++r) {
        const uint32_t h = head0 + 4 * r;
        if (h >= heads) break;
        const float inv = HPW == 1 ? invs : __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(invs), r));
        const bool is_v = h >= num_q_heads + num_kv_heads, use_first = kinds.takes_q_weight(h) == first_q;
        float out[EPL];
#pragma unroll
        for (int j = 0; j < EPL; ++j) {
            float xv = (float)piece[r][j] * inv;
            if (!is_v) xv *= use_first ? first_w[j] : last_w[j];
            asm volatile("" : "+v"(xv));   // the fp32 product is rounded to half, not fused into the conversion
            out[j] = (float)(half_t)xv;
        }
        if (!is_v) {
#pragma unroll
            for (int j = 0; j < EPL; ++j) {
                const uint32_t own = __float_as_uint(out[j]);
                const auto both = __builtin_amdgcn_permlane32_swap(own, own, false, false);      // lanes 0..31 twice, lanes 32..63 twice
                const float x0 = __uint_as_float(both[0]), x1 = __uint_as_float(both[1]);
                float turned = fmaf(x0, x0_by[j], x1 * x1_by[j]);
                asm volatile("" : "+v"(turned));   // an fp32 value before it becomes a half, as above
                out[j] = (lane & 31) * EPL + j < rotated_pairs ? turned : out[j];
            }
        }
        half_t *dst = head_at(h) + lane * EPL;
        if constexpr (VEC) {
            piece_t p;
#pragma unroll
            for (int j = 0; j < EPL; ++j) p[j] = (half_t)out[j];
            *reinterpret_cast<piece_t *>(dst) = p;
        } else {
#pragma unroll
            for (int j = 0; j < EPL; ++j) dst[j] = (half_t)out[j];
        }
    }
}

// any other head_dim: one block per head and token (grid (heads, tokens)): q heads, then k heads, then v heads; token t at position + t
__global__ __launch_bounds__(256) void qkv_epilogue_kernel(half_t *q, half_t *k, half_t *v, const uint16_t *q_weight, const uint16_t *k_weight,
                                                           uint32_t head_dim, uint32_t num_q_heads, uint32_t num_kv_heads, uint32_t position,
                                                           float theta, uint32_t rotated_pairs, float eps, uint32_t q_token_stride,
                                                           uint32_t kv_token_stride) {
    __shared__ half_t normed[kEpilogueMaxHeadDim];
    __shared__ float partial[4];
    const uint32_t hg = blockIdx.x, t = blockIdx.y;
    position += t;
    const bool is_q = hg < num_q_heads, is_k = !is_q && hg < num_q_heads + num_kv_heads;
    half_t *dst = is_q ? q + (size_t)t * q_token_stride + (size_t)hg * head_dim
                       : (is_k ? k + (size_t)t * kv_token_stride + (size_t)(hg - num_q_heads) * head_dim
                               : v + (size_t)t * kv_token_stride + (size_t)(hg - num_q_heads - num_kv_heads) * head_dim);
    const uint16_t *w = is_q ? q_weight : k_weight;
    float acc = 0.0f;
    for (uint32_t i = threadIdx.x; i < head_dim; i += blockDim.x) {
        const float xv = (float)dst[i];
        acc = fmaf(xv, xv, acc);
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = acc;
    __syncthreads();
    const float inv = 1.0f / sqrtf(((partial[0] + partial[1]) + (partial[2] + partial[3])) / (float)head_dim + eps);
    for (uint32_t i = threadIdx.x; i < head_dim; i += blockDim.x) {
        float xv = (float)dst[i] * inv;
        if (is_q || is_k) xv *= bf16_to_f32(w[i]);
        asm volatile("" : "+v"(xv));   // the fp32 product is rounded to half, not fused into the conversion
        normed[i] = (half_t)xv;
    }
    __syncthreads();
    if (!is_q && !is_k) {
        for (uint32_t i = threadIdx.x; i < head_dim; i += blockDim.x) dst[i] = normed[i];
        return;
    }
    const uint32_t half_dim = head_dim / 2;
    for (uint32_t pair = threadIdx.x; pair < half_dim; pair += blockDim.x) {
        float x0 = (float)normed[pair], x1 = (float)normed[half_dim + pair];
        if (pair < rotated_pairs) rope_pair(x0, x1, pair, head_dim, (float)position, theta);
        dst[pair] = (half_t)x0;
        dst[half_dim + pair] = (half_t)x1;
    }
}

int32_t launch_rope(tf_ctx *ctx, tf_stream stream, void *data, uint64_t data_offset, uint32_t position, uint32_t position_step, uint32_t head_dim,
                    uint32_t num_heads, uint32_t num_tokens, uint32_t token_stride, float theta, uint32_t rotated_pairs, const char *who) {
    TF_REQUIRE(ctx, ctx && data, TF_ERR_INVALID_ARGUMENT, "%s: null argument", who);
    TF_REQUIRE(ctx, head_dim % 2 == 0, TF_ERR_INVALID_ARGUMENT, "%s: head_dim must be even", who);
    TF_REQUIRE(ctx, (uint64_t)rotated_pairs * 2 <= head_dim, TF_ERR_INVALID_ARGUMENT, "%s: rotatedPairs * 2 must not exceed head_dim", who);
    TF_REQUIRE(ctx, data_offset % 2 == 0, TF_ERR_INVALID_ARGUMENT, "%s: offsets must be 2-byte aligned", who);
    TF_REQUIRE(ctx, num_heads <= 65535 && num_tokens <= 65535, TF_ERR_INVALID_ARGUMENT, "%s: more than 65535 heads or tokens", who);
    if (rotated_pairs == 0 || num_heads == 0 || num_tokens == 0) return TF_OK;
    const dim3 grid((rotated_pairs + 255) / 256, num_heads, num_tokens);
    hipLaunchKernelGGL(rope_neox_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), reinterpret_cast<half_t *>(at(data, data_offset)),
                       position, position_step, head_dim, token_stride, theta, rotated_pairs);
    return check_launch(ctx, who);
}

int32_t launch_qkv_epilogue(tf_ctx *ctx, tf_stream stream, void *q, uint64_t q_offset, void *k, uint64_t k_offset, void *v, uint64_t v_offset,
                            const void *q_weight, uint64_t q_weight_offset, const void *k_weight, uint64_t k_weight_offset, uint32_t head_dim,
                            uint32_t num_q_heads, uint32_t num_kv_heads, uint32_t position, uint32_t tokens, uint32_t q_token_stride,
                            uint32_t kv_token_stride, float theta, uint32_t rotated_pairs, float eps, const char *who) {
    TF_REQUIRE(ctx, ctx && q && k && v && q_weight && k_weight, TF_ERR_INVALID_ARGUMENT, "%s: null argument", who);
    TF_REQUIRE(ctx, head_dim > 0 && head_dim <= kEpilogueMaxHeadDim, TF_ERR_INVALID_ARGUMENT, "headDim > 512 exceeds the fused QKV epilogue scratch");
    TF_REQUIRE(ctx, head_dim % 2 == 0, TF_ERR_INVALID_ARGUMENT, "%s: head_dim must be even", who);
    TF_REQUIRE(ctx, (uint64_t)rotated_pairs * 2 <= head_dim, TF_ERR_INVALID_ARGUMENT, "rotatedPairs must fit inside one NeoX head");
    TF_REQUIRE(ctx, q_offset % 2 == 0 && k_offset % 2 == 0 && v_offset % 2 == 0 && q_weight_offset % 2 == 0 && k_weight_offset % 2 == 0,
               TF_ERR_INVALID_ARGUMENT, "%s: offsets must be 2-byte aligned", who);
    TF_REQUIRE(ctx, tokens <= 65535, TF_ERR_INVALID_ARGUMENT, "%s: more than 65535 tokens", who);
    const uint32_t groups = num_q_heads + 2 * num_kv_heads;
    if (groups == 0 || tokens == 0) return TF_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    half_t *qp = reinterpret_cast<half_t *>(at(q, q_offset)), *kp = reinterpret_cast<half_t *>(at(k, k_offset)), *vp = reinterpret_cast<half_t *>(at(v, v_offset));
    const uint16_t *qw = reinterpret_cast<const uint16_t *>(at(q_weight, q_weight_offset)), *kw = reinterpret_cast<const uint16_t *>(at(k_weight, k_weight_offset));
    if (head_dim == 64 || head_dim == 128 || head_dim == 256 || head_dim == 512) {
        // several heads a wave once the blocks fill the chip eight deep: the angles are shared by more heads
        const uint64_t quads = (uint64_t)tokens * ((groups + 3) / 4);
        const uint32_t per_wave = quads >= 8 * kEpilogueBlocks ? 8u : quads >= 4 * kEpilogueBlocks ? 4u : quads >= 2 * kEpilogueBlocks ? 2u : 1u;
        const dim3 grid((groups + 4 * per_wave - 1) / (4 * per_wave), tokens);
        const unsigned piece = head_dim / 64 * 2;
        const bool vec = aligned(qp, piece) && aligned(kp, piece) && aligned(vp, piece) && q_token_stride * 2 % piece == 0 && kv_token_stride * 2 % piece == 0;
        auto launch = [&](auto epl, auto vectors) {
            auto with = [&](auto heads) {
                hipLaunchKernelGGL((qkv_epilogue_wave_kernel<decltype(epl)::value, decltype(vectors)::value, decltype(heads)::value>), grid, dim3(256), 0, st, qp, kp, vp, qw,
                                   kw, num_q_heads, num_kv_heads, position, theta, rotated_pairs, eps, q_token_stride, kv_token_stride);
            };
            per_wave == 8 ? with(std::integral_constant<int, 8>{}) : per_wave == 4 ? with(std::integral_constant<int, 4>{})
            : per_wave == 2 ? with(std::integral_constant<int, 2>{}) : with(std::integral_constant<int, 1>{});
        };
        auto either = [&](auto epl) { vec ? launch(epl, std::true_type{}) : launch(epl, std::false_type{}); };
        switch (head_dim) {
            case 64: launch(std::integral_constant<int, 1>{}, std::true_type{}); break;
            case 128: either(std::integral_constant<int, 2>{}); break;
            case 256: either(std::integral_constant<int, 4>{}); break;
            default: either(std::integral_constant<int, 8>{}); break;
        }
        return check_launch(ctx, who);
    }
    hipLaunchKernelGGL(qkv_epilogue_kernel, dim3(groups, tokens), dim3(256), 0, st, qp, kp, vp, qw, kw, head_dim, num_q_heads, num_kv_heads, position, theta,
                       rotated_pairs, eps, q_token_stride, kv_token_stride);
    return check_launch(ctx, who);
}

}  // namespace

extern "C" {

int32_t tf_rope_default_neox(tf_ctx *ctx, tf_stream stream, void *data, uint64_t data_offset, uint32_t position, uint32_t head_dim,
                             uint32_t num_heads, uint32_t num_tokens, float theta) {
    return launch_rope(ctx, stream, data, data_offset, position, 0, head_dim, num_heads, num_tokens, num_heads * head_dim, theta, head_dim / 2,
                       "rope_default_neox");
}

int32_t tf_rope_proportional_neox(tf_ctx *ctx, tf_stream stream, void *data, uint64_t data_offset, uint32_t position, uint32_t head_dim,
                                  uint32_t num_heads, uint32_t num_tokens, uint32_t rotated_pairs, float theta) {
    return launch_rope(ctx, stream, data, data_offset, position, 0, head_dim, num_heads, num_tokens, num_heads * head_dim, theta, rotated_pairs,
                       "rope_proportional_neox");
}

int32_t tf_prefill_rope_default_neox_block(tf_ctx *ctx, tf_stream stream, void *data, uint64_t data_offset, uint32_t start_position,
                                           uint32_t query_count, uint32_t head_dim, uint32_t num_heads, uint32_t token_stride_elements, float theta) {
    TF_REQUIRE(ctx, ctx != nullptr, TF_ERR_INVALID_ARGUMENT, "prefill_rope_default_neox_block: null context");
    TF_REQUIRE(ctx, query_count > 0, TF_ERR_INVALID_ARGUMENT, "queryCount must be positive");
    TF_REQUIRE(ctx, (uint64_t)token_stride_elements >= (uint64_t)num_heads * head_dim, TF_ERR_INVALID_ARGUMENT, "token stride is too small");
    return launch_rope(ctx, stream, data, data_offset, start_position, 1, head_dim, num_heads, query_count, token_stride_elements, theta, head_dim / 2,
                       "prefill_rope_default_neox_block");
}

int32_t tf_prefill_rope_proportional_neox_block(tf_ctx *ctx, tf_stream stream, void *data, uint64_t data_offset, uint32_t start_position,
                                                uint32_t query_count, uint32_t head_dim, uint32_t num_heads, uint32_t rotated_pairs,
                                                uint32_t token_stride_elements, float theta) {
    TF_REQUIRE(ctx, ctx != nullptr, TF_ERR_INVALID_ARGUMENT, "prefill_rope_proportional_neox_block: null context");
    TF_REQUIRE(ctx, query_count > 0, TF_ERR_INVALID_ARGUMENT, "queryCount must be positive");
    TF_REQUIRE(ctx, (uint64_t)token_stride_elements >= (uint64_t)num_heads * head_dim, TF_ERR_INVALID_ARGUMENT, "token stride is too small");
    return launch_rope(ctx, stream, data, data_offset, start_position, 1, head_dim, num_heads, query_count, token_stride_elements, theta, rotated_pairs,
                       "prefill_rope_proportional_neox_block");
}

int32_t tf_fused_qkv_epilogue(tf_ctx *ctx, tf_stream stream, void *q, uint64_t q_offset, void *k, uint64_t k_offset, void *v, uint64_t v_offset,
                              const void *q_weight, uint64_t q_weight_offset, const void *k_weight, uint64_t k_weight_offset, uint32_t head_dim,
                              uint32_t num_q_heads, uint32_t num_kv_heads, uint32_t position, float theta, uint32_t rotated_pairs, float eps) {
    return launch_qkv_epilogue(ctx, stream, q, q_offset, k, k_offset, v, v_offset, q_weight, q_weight_offset, k_weight, k_weight_offset, head_dim,
                               num_q_heads, num_kv_heads, position, 1, 0, 0, theta, rotated_pairs, eps, "fused_qkv_epilogue");
}

int32_t tf_prefill_qkv_epilogue_block(tf_ctx *ctx, tf_stream stream, void *q, uint64_t q_offset, void *k, uint64_t k_offset, void *v,
                                      uint64_t v_offset, const void *q_weight, uint64_t q_weight_offset, const void *k_weight,
                                      uint64_t k_weight_offset, uint32_t start_position, uint32_t query_count, uint32_t head_dim,
                                      uint32_t num_q_heads, uint32_t num_kv_heads, uint32_t q_token_stride_elements,
                                      uint32_t kv_token_stride_elements, float theta, uint32_t rotated_pairs, float eps) {
    TF_REQUIRE(ctx, ctx != nullptr, TF_ERR_INVALID_ARGUMENT, "prefill_qkv_epilogue_block: null context");
    // PrefillQKVEpilogue.encode's preconditions (PrefillQKVEpilogue.swift:34-43)
    TF_REQUIRE(ctx, query_count > 0, TF_ERR_INVALID_ARGUMENT, "queryCount must be positive");
    TF_REQUIRE(ctx, head_dim > 0 && head_dim % 2 == 0, TF_ERR_INVALID_ARGUMENT, "headDim must be positive and even");
    TF_REQUIRE(ctx, num_q_heads > 0, TF_ERR_INVALID_ARGUMENT, "numQHeads must be positive");
    TF_REQUIRE(ctx, num_kv_heads > 0, TF_ERR_INVALID_ARGUMENT, "numKVHeads must be positive");
    TF_REQUIRE(ctx, rotated_pairs > 0, TF_ERR_INVALID_ARGUMENT, "rotatedPairs must be positive");
    TF_REQUIRE(ctx, (uint64_t)rotated_pairs * 2 <= head_dim, TF_ERR_INVALID_ARGUMENT, "rotatedPairs must fit inside one head");
    TF_REQUIRE(ctx, (uint64_t)q_token_stride_elements >= (uint64_t)num_q_heads * head_dim, TF_ERR_INVALID_ARGUMENT, "Q token stride is too small");
    TF_REQUIRE(ctx, (uint64_t)kv_token_stride_elements >= (uint64_t)num_kv_heads * head_dim, TF_ERR_INVALID_ARGUMENT, "KV token stride is too small");
    return launch_qkv_epilogue(ctx, stream, q, q_offset, k, k_offset, v, v_offset, q_weight, q_weight_offset, k_weight, k_weight_offset, head_dim,
                               num_q_heads, num_kv_heads, start_position, query_count, q_token_stride_elements, kv_token_stride_elements, theta,
                               rotated_pairs, eps, "prefill_qkv_epilogue_block");
}

}  // extern "C"
