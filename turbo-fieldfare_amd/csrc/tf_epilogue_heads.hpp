// Numbering of the heads in the fused per-head norm and RoPE step: q heads, then k heads, then v heads.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define TF_HEADS_FN __host__ __device__ __forceinline__
#else
#define TF_HEADS_FN inline
#endif

namespace tfk {

struct EpilogueHeads {
    uint32_t q, kv;
    TF_HEADS_FN uint32_t count() const { return q + 2 * kv; }
    // Waves are launched in fours and look one round ahead, so some ask for heads past the last; they are given the last head's
    // data and use none of it.
    TF_HEADS_FN uint32_t read(uint32_t h) const { return h < count() ? h : count() - 1; }
    // Which weight row a wave asks for with its head (v heads ask for one they do not use).  Without k and v heads the k weight
    // is never touched: a caller may have none.
    TF_HEADS_FN bool takes_q_weight(uint32_t h) const { return read(h) < q; }
};

}  // namespace tfk
