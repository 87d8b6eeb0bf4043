// Shared pieces of the prefill / multi-token path: POD layouts, expert lookup, work lists.
#pragma once

#include "tf_gemv_kernels.hpp"
#include "tf_qmm.hpp"

namespace tfk {

// Where the expert blobs live: a table of up to 16 (id, pointer) bindings — the reference's streamed tile
// (PrefillGroupedRoutedMoE.swift:185-216) — or a resident pool indexed by expert id.
struct ExpertTable {
    const uint8_t *blob[TF_MAX_TILE_EXPERTS];
    uint32_t local_id[TF_MAX_TILE_EXPERTS];
    uint32_t live;
    const uint8_t *pool;
    uint64_t stride;
    uint32_t num_experts;
};

// nullptr when the expert is not bound in the tile (the reference's kernels skip such pairs, prefill.metal:611-618).
__device__ __forceinline__ const uint8_t *expert_base(const ExpertTable &t, uint32_t expert) {
    if (t.pool) {
        const uint32_t e = expert < t.num_experts ? expert : t.num_experts - 1;
        return t.pool + (uint64_t)e * t.stride;
    }
    for (uint32_t s = 0; s < t.live; ++s)
        if (t.local_id[s] == expert) return t.blob[s];
    return nullptr;
}

// Work list: runs of sorted pairs that share one expert, each at most kChunkPairs long.  Either a short list passed with
// the kernel arguments or a device array written by the grouping kernel (with its length in device memory).
constexpr uint32_t kChunkPairs = 128;
constexpr uint32_t kInlineChunks = 48;
struct ChunkList {
    uint32_t n;
    tf_prefill_group inline_chunks[kInlineChunks];
    const tf_prefill_group *dev;
    const uint32_t *dev_n;
};

__device__ __forceinline__ bool get_chunk(const ChunkList &cl, uint32_t i, tf_prefill_group &out) {
    if (cl.dev) {
        if (i >= *cl.dev_n) return false;
        out = cl.dev[i];
    } else {
        if (i >= cl.n) return false;
        out = cl.inline_chunks[i];
    }
    return true;
}

// A shared expert's block of rows riding along in the launches of the grouped matrix-core kernels: its gate / up / GeGLU
// tiles ahead of the grouped gate / up tiles, its down tiles ahead of the grouped down tiles.
struct DenseRide {
    const tf_projection *gate, *up, *down;
    const half_t *x;      // [rows, gate->cols], row stride ldx halves
    long ldx;
    half_t *acts;         // [rows, gate->rows] activations between the two launches
    half_t *y;            // [rows, down->rows], row stride ldy halves
    long ldy;
    int rows;
    bool split;           // gate / up as launch_geglu_split computes them, down as qmm_split_variant says
    bool slice;           // both as the slice kernels compute them (neither: the dense tiles)
};

// Up to here the shared expert's gate / up and down are computed as the split kernels do: in launches of their own beside the quad kernels (53
// rows of 2112 x 2816: 20 us for both against 50 on the dense tiles), or riding in the routed tiles' launches (the one call, 53 rows, 16 experts
// of 704 x 2816: 47 us against 56 with dense tiles riding; 32 experts 57 against 58, 64 experts 71 against 75).  The rule asks for the rows
// alone, never for the experts: the shared expert by itself and the one call give the same bits.
constexpr uint32_t kSharedSplitMaxRows = 79;
// From there to here as the slice kernels do, whose shape allows it: in launches of their own (2112 x 2816, 96 / 128 / 200 / 256 rows: 54 / 59 / 62 / 60 us
// on the dense tiles, 27 / 29 / 35 / 38 so; up to 79 rows 20 - 22 split, 19 - 26 so), or by some of the blocks of the routed slice launches.
// The last row of that range depends on the columns: of 2560 and fewer, 200 to 256 tokens are no faster with both in slice launches than with both on the
// tiles, and slower where experts are popular (128 experts, equally popular and popular, one call with a shared expert, tiles/slices, us: 1280 x 640
// 200 tokens 69/69 52/53, 256 69/73 52/63; 2048 x 768 120/111 74/76, 122/119 75/86; 2560 x 640 134/119 71/78, 133/127 82/92; but 144 tokens
// 69/65 50/47, 119/100 67/61, 136/110 70/66).  At 2816 x 704 163/134 88/88 and 166/142 90/102; rows with a common direction, routed stages, 200 tokens 129/106.
constexpr uint32_t kSliceWideCols = 2688;
inline uint32_t slice_max_rows(uint32_t cols) { return cols >= kSliceWideCols ? 256u : 192u; }
constexpr uint32_t kSliceMinExperts = 48;      // of the routed stages, up to kSharedSplitMaxRows tokens (run_grouped)

// Operands of the grouped expert stages, as the launch helpers pass them on.
struct GroupedGeom {
    const tf_prefill_pair *pairs;
    const half_t *hidden;
    long hidden_stride;
    half_t *acts;
    uint32_t acts_pair_base;
    half_t *route_partials;
    int d, f, top_k;
};

// The quad kernels (tf_prefill_quad.hip): grouped gate / up / GeGLU and down for chunks of a few pairs, weights streamed once per
// expert.  kQuadMaxD / kQuadMaxF: the widest rows they take; the caller checks alignment and shape (run_grouped).
constexpr int kQuadMaxD = 3072, kQuadMaxF = 1024;
int32_t launch_grouped_quad(tf_ctx *ctx, hipStream_t st, const ExpertTable &tab, const tf_expert_offsets &off, const ChunkList &cl,
                            uint32_t n_chunks_upper, const GroupedGeom &g, tf_dtype sd, uint32_t stream_pairs);

// The slice kernels (tf_prefill_slice.hip): the same stages for chunks of a few dozen pairs, activations in registers.
bool grouped_slice_ok(const ExpertTable &tab, const ChunkList &cl, uint32_t pair_count, int d, int f);
int32_t launch_grouped_slice(tf_ctx *ctx, hipStream_t st, const ExpertTable &tab, const tf_expert_offsets &off, const ChunkList &cl,
                             uint32_t n_chunks_upper, const GroupedGeom &g, tf_dtype sd, const DenseRide *ride);
// and a shared expert's block of rows, in launches of its own or (ride above) beside the routed pairs
bool shared_slice_ok(const tf_projection *gate);
int32_t launch_shared_slice(tf_ctx *ctx, hipStream_t st, const DenseRide &ride, tf_dtype sd);

// Dense products whose waves split the contraction (tf_qmm_split.hip).  qmm_split_variant: kSplitNone where the 128 x 256 tiles are the
// better kernel, otherwise what launch_qmm_split is to be given; operands as qmm_operands_ok() demands.
enum { kSplitNone = 0, kSplit32x32, kSplit64x32, kSplit64x64 };
int qmm_split_variant(int m, int n, int k, long ldx, int num_cus);
int32_t launch_qmm_split(tf_ctx *ctx, hipStream_t st, int variant, const uint8_t *w, const uint8_t *s, const uint8_t *b, const half_t *x, long ldx,
                         half_t *y, long ldy, int m, int n, int k, tf_dtype sd);
// the same for a gate and an up matrix with GeGLU (rows of up to 4096 columns either way, so that the result can also be had inside a grouped launch)
bool geglu_split_ok(const tf_projection *gate, long ldx);
int32_t launch_geglu_split(tf_ctx *ctx, hipStream_t st, const tf_projection *gate, const tf_projection *up, const half_t *x, long ldx, half_t *a_out,
                           long lda, int m, tf_dtype sd);

bool shared8_split_ok(const tf_projection *gate, long ldx);
int32_t launch_shared8_split(tf_ctx *ctx, hipStream_t st, const tf_projection *gate, const tf_projection *up, const tf_projection *down, const half_t *x,
                             long ldx, half_t *acts, half_t *y, long ldy, int m, tf_dtype sd);

}  // namespace tfk
