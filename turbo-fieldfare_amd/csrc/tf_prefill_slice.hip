// Grouped expert stages for blocks of tokens whose experts see a few to a few dozen pairs: the slice kernels.
#include <algorithm>

#include "tf_prefill_kernels.hpp"

using namespace tfk;

namespace {

// Every touched expert streams through once, at the rate of a plain read; the arithmetic has to fit beside it.
//
// A wave keeps the activations of up to 32 pairs over a SLICE of the contraction (four quantization groups, 256 columns) in registers, as
// the A operands of v_mfma_f32_32x32x16_f16, for as long as its block works on these pairs.  Weight rows pass by it, 32 at a time: 128
// bytes of each, the lines that its slice covers, come through a wave-private ring in LDS (two tiles deep, copied by the load unit: nothing but
// whole 128-byte lines is asked for, and no register waits for memory), and nibbles masked out of the words are the B operand as they are:
// read as fp16 subnormals they are exactly q 2^-24.  (Every word is shifted for each of its four masks.  With two masks fewer shifts, 16 q against
// activations of a sixteenth, activations below 2^-10 lose up to four bits: at 1e-4 0.6 % of the result.  The shifts cost 1 %: both launches of 128 / 256
// tokens 110.6 / 120.8 -> 111.7 / 121.3 us.)  A group's four instructions start from zero; their sums are then multiplied by the
// row's scale in fp32, and the bias terms of a slice are one more instruction: bias times the sums of the activations, those split into three
// bf16 parts, exact.  So a weight is q s + b in 32 bits, as in the quad kernels, and a 32 x 64 piece of weights costs 28 + NR vector
// instructions against the 64 that rounding it to fp16 takes in the tile kernels.  The sums of subnormal operands come out with
// an error of 2e-6 to 7e-6 of the outputs' norm (against 64-bit sums; those of the quad kernels likewise).
//
// A row's slices lie with different waves: SLICES of them (11 at 2816 columns) share a tile, their sums meet in LDS and are added in slice
// order; with few slices (3 at 704 columns) a block holds several such groups of waves, each on tiles of its own.  One block of up to twelve
// waves to a compute unit.
//
// The work of a launch is cut into units: up to 32 pairs of one chunk against all of its expert's rows.  The units' tiles are dealt out to the
// blocks by what they cost; where a block's share crosses into the next unit, the weights of that unit are already on their way.  A
// shared expert's block of rows is one more list of a single chunk, of rows that are their own tokens: some of the blocks take that.
//
// Measured (128 experts of 704 x 2816, 128 tokens with a common direction, both launches 111 -> 90 us against the tiles, 53 tokens 104 -> 75
// against the quad kernels; as of then, exact small activations and infinities cost 2 % of that since).  What bounds them: in the middle of a launch 45 KB of
// weights and 6 KB of scales a compute unit every 2.3 us are asked for, 5.6 TB/s by that count, two tiles of each wave on their way; the adding up of the
// sums, when one wave did all of it, made that 2.6.  A launch's first tile is done 11 to 12 us after its start (work list 2, pairs 2, activations 2, the
// first weights of all units at once 4): what is left.  Over a whole gate / up launch with a shared expert (128 tokens, 61 us) the counters have 112 MB from
// memory, vector instructions in 41 % of the issue slots, the matrix units busy for 22 %.
constexpr int kSliceGroups = 4;                  // quantization groups of a slice
constexpr int kSliceMaxWaves = 12;
constexpr uint32_t kSliceBatch = 32;             // pairs of a unit
constexpr uint32_t kSliceWBytes = 32 * 128;      // one wave's weights of a tile
constexpr uint32_t kSliceSlot = kSliceWBytes + 512;      // and its scales and biases, eight bytes a row each
constexpr int kSliceCopies = 6;                  // requests a tile
constexpr uint32_t kSliceSums = 64 * 16 * 4;     // one wave's sums of a tile; half of it twice where they fit in half
constexpr int kSliceListRounds = 4;              // the work list is looked at 64 chunks at a time, four times 64 in one trip to memory; the table holds as many
constexpr uint32_t kSliceList = 64 * kSliceListRounds;
constexpr uint32_t kSliceRing = 0, kSliceSumsAt = kSliceMaxWaves * 2 * kSliceSlot, kSliceTableAt = kSliceSumsAt + kSliceMaxWaves * kSliceSums,
                   kSliceRowsAt = kSliceTableAt + 3 * 4 * kSliceList, kSlicePairsAt = kSliceRowsAt + 4 * kSliceBatch, kSliceLds = kSlicePairsAt + 16 * kSliceBatch;
static_assert(kSliceLds <= 160 * 1024, "one block a compute unit");

// What a position costs with up to 8, up to 16 and up to 32 pairs (gate / up 2.33, 2.5 and 2.85 us), and what the change to another unit
// costs, its first tile's.
__host__ __device__ constexpr uint32_t slice_tile_cost(uint32_t pairs) { return pairs <= 8u ? 8u : pairs <= 16u ? 9u : 10u; }
constexpr uint32_t kSliceUnitCost = 10;
__host__ __device__ constexpr uint32_t slice_unit_cost(uint32_t pairs, uint32_t positions) { return kSliceUnitCost + slice_tile_cost(pairs) * positions; }

struct SliceProblem {
    const uint8_t *w[2], *s[2], *b[2];           // gate and up, or down twice; of expert 0 where there are several
    uint64_t stride;                             // from one expert to the next
    const half_t *x;                             // rows of activations: of tokens, or of pairs
    long x_stride;
    half_t *out;
    long out_stride;
    int k, n;
    int slices, row_groups;
};
struct SliceArgs {
    SliceProblem routed, shared;
    const tf_prefill_group *list;
    const uint32_t *list_count;
    uint32_t list_cap, num_experts;              // list_cap == 0: no routed pairs
    const tf_prefill_pair *pairs;
    uint32_t pair_base, top_k;
    uint32_t shared_rows;                        // 0: no shared expert
};

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// 16 or 4 bytes a lane from `from` (a lane's own) straight into LDS: lane l's land at to + 16 l or to + 4 l
typedef const __attribute__((address_space(1))) void *global_ptr;
typedef __attribute__((address_space(3))) void *lds_ptr;
__device__ __forceinline__ void slice_copy16(const void *from, uint32_t to) { __builtin_amdgcn_global_load_lds((global_ptr)(uintptr_t)from, (lds_ptr)(uintptr_t)to, 16, 0, 0); }
__device__ __forceinline__ void slice_copy4(const void *from, uint32_t to) { __builtin_amdgcn_global_load_lds((global_ptr)(uintptr_t)from, (lds_ptr)(uintptr_t)to, 4, 0, 0); }
__device__ __forceinline__ void lds_put16(uint32_t addr, f32x4 v) { asm volatile("ds_write_b128 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
__device__ __forceinline__ void lds_put4(uint32_t addr, uint32_t v) { asm volatile("ds_write_b32 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
// What has been written to LDS is there for the block; requests to memory stay on their way.
__device__ __forceinline__ void slice_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void stay_in_order() { asm volatile("" ::: "memory"); }      // requests are counted when they are waited for

__device__ __forceinline__ uint32_t slice_running_sum(uint32_t v) {      // lane l: the sum over lanes 0 .. l
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);
    return v;
}
__device__ __forceinline__ uint32_t slice_chunk_cost(uint32_t pairs, uint32_t positions) {
    const uint32_t whole = pairs / kSliceBatch, rest = pairs - whole * kSliceBatch;
    return whole * slice_unit_cost(kSliceBatch, positions) + (rest ? slice_unit_cost(rest, positions) : 0u);
}

// The sixteen sums of a lane, one tile: 32 weight rows (the lane's row is lane & 31) against pairs acc_row(r, lane), of which the first
// NR sums (2 NR pairs) are wanted.  x: the wave's activations, xs: the parts of their sums.  Units of 2^-24.
// ODD: the pairs of the lanes with lane_odd have infinities or NaN among these activations (and zeros for xs).  Their sums are taken over the weights
// themselves, rounded to fp16 as the tile kernels do: infinities of the sign that weight and activation give, where q s and b apart would give NaN (a nibble
// of zero, the parts of an infinite sum).  The other pairs' are the same as ever.
template <int SD, int NR, bool ODD>
__device__ __forceinline__ void slice_multiply(const half8_t (&x)[kSliceGroups][4], const bf16x8_t xs, const u32x4 (&w)[kSliceGroups], u32x2 s, u32x2 b,
                                               bool lane_odd, float16_t &acc) {
    float16_t zero;
#pragma unroll
    for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
    acc = zero;
    auto masked = [&](const half8_t row, bool of_odd) {                  // zeros for the pairs of the other kind
        u32x4 v = __builtin_bit_cast(u32x4, row);
        asm volatile("" : "+v"(v));              // made here, again for every tile
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = lane_odd == of_odd ? v[j] : 0u;
        return __builtin_bit_cast(half8_t, v);
    };
    if constexpr (ODD) {
#pragma unroll
        for (int g = 0; g < kSliceGroups; ++g) {
            const uint32_t s16 = (g & 1) ? s[g >> 1] >> 16 : s[g >> 1] & 0xFFFFu, b16 = (g & 1) ? b[g >> 1] >> 16 : b[g >> 1] & 0xFFFFu;
            const float sc = sb_to_f32<SD>((uint16_t)s16), bias = sb_to_f32<SD>((uint16_t)b16);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                uint32_t word = w[g][d];
                asm volatile("" : "+v"(word));   // as below
                half8_t weight;
#pragma unroll
                for (int j = 0; j < 8; ++j)      // (a weight beyond fp16 stays finite: the other pairs' zeros meet it too)
                    weight[j] = (half_t)fminf(fmaxf(fmaf((float)(word >> (4 * (j >> 1) + 16 * (j & 1)) & 15u), sc, bias), -65504.0f), 65504.0f);
                asm volatile("" : "+v"(weight));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(masked(x[g][d], true), weight, acc, 0, 0, 0);
            }
            asm volatile("" : "+v"(s), "+v"(b));
        }
    }
    if constexpr (SD == 0) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xs, __builtin_bit_cast(bf16x8_t, u32x4{b[0], b[1], b[0], b[1]}), acc, 0, 0, 0);
    } else {
        // an fp16 bias is the sum of two bf16 numbers, of its upper eight and its lower three bits
        u32x2 hi, lo;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float b0 = f16_to_f32((uint16_t)(b[j] & 0xFFFFu)), b1 = f16_to_f32((uint16_t)(b[j] >> 16));
            const uint32_t h0 = __float_as_uint(b0) & 0xFFFF0000u, h1 = __float_as_uint(b1) & 0xFFFF0000u;
            hi[j] = (h0 >> 16) | h1;
            lo[j] = (__float_as_uint(b0 - __uint_as_float(h0)) >> 16) | (__float_as_uint(b1 - __uint_as_float(h1)) & 0xFFFF0000u);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xs, __builtin_bit_cast(bf16x8_t, u32x4{lo[0], lo[1], lo[0], lo[1]}), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xs, __builtin_bit_cast(bf16x8_t, u32x4{hi[0], hi[1], hi[0], hi[1]}), acc, 0, 0, 0);
    }
#pragma unroll
    for (int g = 0; g < kSliceGroups; ++g) {
        float16_t c = zero;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            uint32_t word = w[g][d];
            asm volatile("" : "+v"(word));       // the operands are made here, word by word: all of a tile's at once would not fit the registers
            const u32x4 q = {word & 0x000F000Fu, word >> 4 & 0x000F000Fu, word >> 8 & 0x000F000Fu, word >> 12 & 0x000F000Fu};
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ODD ? masked(x[g][d], false) : x[g][d], __builtin_bit_cast(half8_t, q), c, 0, 0, 0);
        }
        const uint32_t sv = s[g >> 1];
        const float sc = SD == 0 ? __uint_as_float((g & 1) ? sv & 0xFFFF0000u : sv << 16) : f16_to_f32((uint16_t)((g & 1) ? sv >> 16 : sv & 0xFFFFu));
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[r] = fmaf(sc, c[r], acc[r]);
    }
}

// LONG: the work list has room for more chunks than the table.  A share of such a list is found by a walk over it, and chunks beyond the table come from
// memory.  Which of the two it is never shows in the results; both launches of 128 tokens (128 experts) 118 / 111 us and, from a list with room for 400 chunks
// that has no more than the other, 119 / 111; of 80 tokens 104 / 108.
template <bool GATE_UP, int SD, bool LONG>
__global__ __launch_bounds__(64 * kSliceMaxWaves) void grouped_slice_kernel(SliceArgs a) {
    constexpr int kRows = GATE_UP ? 16 : 32;           // output columns of a tile: 16 of gate with the same 16 of up, or 32
    __shared__ __align__(128) uint8_t lds_area[kSliceLds];
    const uint32_t lds = (uint32_t)(uintptr_t)lds_area, table = lds + kSliceTableAt;
    const int lane = threadIdx.x & 63, wave = uniform_int((int)(threadIdx.x >> 6));
    const int i = lane & 31, kb = lane >> 5;
    auto positions_of = [&](const SliceProblem &p) { return ((uint32_t)(p.n / kRows) + (uint32_t)p.row_groups - 1) / (uint32_t)p.row_groups; };

    // ---- the work list: for every chunk the cost of those before it, where its pairs start, its expert and how many pairs it has
    uint32_t n_chunks = 0u, cost = 0u;                 // cost: of all units
    const uint32_t routed_positions = a.list_cap != 0u ? positions_of(a.routed) : 0u;
    tf_prefill_group mine[kSliceListRounds];           // a lane's of the kSliceList chunks in hand
    uint32_t through[kSliceListRounds], own_cost[kSliceListRounds];
    auto take_chunks = [&](uint32_t from) {
#pragma unroll
        for (int r = 0; r < kSliceListRounds; ++r) mine[r] = a.list[min(from + 64u * r + (uint32_t)lane, a.list_cap - 1u)];      // no branch: one trip to memory
    };
    auto add_costs = [&](uint32_t from) {
#pragma unroll
        for (int r = 0; r < kSliceListRounds; ++r) {
            own_cost[r] = from + 64u * r + (uint32_t)lane < n_chunks ? slice_chunk_cost(mine[r].pair_count, routed_positions) : 0u;
            through[r] = cost + slice_running_sum(own_cost[r]);
            cost = (uint32_t)__builtin_amdgcn_readlane((int)through[r], 63);
        }
    };
    if (a.list_cap != 0u) {
        take_chunks(0u);
        n_chunks = uniform_u32(min(*a.list_count, a.list_cap));
    }
    add_costs(0u);
    if constexpr (LONG)
        for (uint32_t from = kSliceList; from < n_chunks; from += kSliceList) {
            take_chunks(from);
            add_costs(from);
        }
    // ---- the block's part: neighbours in the order of the work sit on one XCD, so that the units of a popular expert find its rows in one L2
    const uint32_t blocks = gridDim.x;
    uint32_t block = (blocks & 7u) == 0u ? (blockIdx.x & 7u) * (blocks >> 3) + (blockIdx.x >> 3) : blockIdx.x, of = blocks;
    bool shared = false;
    if (a.shared_rows != 0u) {
        const uint64_t cs = slice_chunk_cost(a.shared_rows, positions_of(a.shared)), cr = cost;
        const uint32_t for_shared = cr == 0u ? blocks : min(max((uint32_t)((blocks * cs + (cs + cr) / 2u) / (cs + cr)), 1u), max(blocks - 1u, 1u));
        shared = block < for_shared;
        of = shared ? for_shared : blocks - for_shared;
        block -= shared ? 0u : for_shared;
        if (shared) {
            n_chunks = 1u;
            cost = (uint32_t)cs;
        }
    }
    const SliceProblem p = shared ? a.shared : a.routed;
    const uint32_t positions = positions_of(p);
    struct Place {
        uint32_t chunk, batch, tile;
    };
    // If the tile at which `spent` of all units' cost is behind belongs to one of 64 chunks, a lane each, from `base` on: into `at`
    auto place_among = [&](uint32_t spent, uint32_t base, uint32_t cost_before, uint32_t chunk_pairs, Place &at) {
        const uint64_t owners = __ballot(spent - cost_before < slice_chunk_cost(chunk_pairs, positions));      // wraps far beyond for a chunk that comes later
        if (owners == 0ull) return false;
        const int owner = (int)__builtin_ctzll(owners);
        const uint32_t pairs = (uint32_t)__builtin_amdgcn_readlane((int)chunk_pairs, owner), whole = slice_unit_cost(kSliceBatch, positions);
        uint32_t rest = spent - (uint32_t)__builtin_amdgcn_readlane((int)cost_before, owner);
        at.chunk = base + (uint32_t)owner;
        at.batch = min(rest / whole, (pairs - 1u) / kSliceBatch);
        rest -= at.batch * whole;
        at.tile = (rest > kSliceUnitCost ? rest - kSliceUnitCost : 0u) / slice_tile_cost(min(pairs - at.batch * kSliceBatch, kSliceBatch));
        return true;
    };
    Place first, last;                                 // the block's first tile, and the one behind its last
    uint32_t table_from = 0u;                          // the table holds the chunks from here on: all of them, or (LONG) those from the block's first on
    auto share_at = [&](uint32_t i) { return (uint32_t)((uint64_t)cost * (block + i) / of); };
    bool placed = false;
    if constexpr (LONG)
        if (n_chunks > kSliceList) {
            const uint32_t from_cost = share_at(0u), to_cost = share_at(1u);
            first = last = Place{n_chunks, 0u, 0u};
            bool found_first = from_cost >= cost, found_last = to_cost >= cost;
            cost = 0u;
            for (uint32_t from = 0u; from < n_chunks && !(found_first && found_last); from += kSliceList) {
                take_chunks(from);
                add_costs(from);
#pragma unroll
                for (int r = 0; r < kSliceListRounds; ++r) {
                    const uint32_t pairs = from + 64u * r + (uint32_t)lane < n_chunks ? mine[r].pair_count : 0u;
                    if (!found_first) found_first = place_among(from_cost, from + 64u * r, through[r] - own_cost[r], pairs, first);
                    if (!found_last) found_last = place_among(to_cost, from + 64u * r, through[r] - own_cost[r], pairs, last);
                }
            }
            table_from = first.chunk;
            take_chunks(table_from);
            placed = true;
        }
    auto packed = [&](const tf_prefill_group &chunk) { return min(chunk.expert, a.num_experts - 1u) << 16 | chunk.pair_count; };
    if (wave == 0) {
#pragma unroll
        for (int r = 0; r < kSliceListRounds; ++r) {
            const uint32_t entry = table + 4u * (64u * r + (uint32_t)lane);
            const bool there = table_from + 64u * r + (uint32_t)lane < n_chunks;
            lds_put4(entry, shared ? 0u : through[r] - own_cost[r]);       // where all chunks are here
            lds_put4(entry + 4u * kSliceList, shared ? 0u : mine[r].pair_start);
            lds_put4(entry + 8u * kSliceList, !there ? 0u : shared ? a.shared_rows : packed(mine[r]));
        }
    }
    slice_barrier();

    const int groups = p.k >> 6;
    const uint32_t row_bytes = (uint32_t)p.k >> 1, sb_row_bytes = (uint32_t)groups * 2u;
    const int rg = wave / p.slices, slice = wave - rg * p.slices;
    const bool working = rg < p.row_groups;            // a wave without a slice keeps the others company at their barriers
    // the last slice of a row starts early enough to be whole; its first `skip` groups are the slice before's (activations of zero here)
    const int g0 = min(kSliceGroups * slice, groups - kSliceGroups), skip = kSliceGroups * slice - g0;
    const uint32_t tiles = (uint32_t)(p.n / kRows);

    struct Unit {
        uint32_t chunk, batch;                         // batch: of the chunk's
        uint32_t expert, first, count, after;          // its pairs; those of the chunk behind them
    };
    auto unit_of = [&](uint32_t chunk, uint32_t batch) {
        uint32_t start, what;
        if (!LONG || chunk - table_from < kSliceList) {
            asm volatile("ds_read_b32 %0, %2 offset:%3\n\tds_read_b32 %1, %2 offset:%4\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(start), "=&v"(what) : "v"(table + 4u * (chunk - table_from)), "n"(4 * kSliceList), "n"(8 * kSliceList) : "memory");
        } else {                                           // a share of more than kSliceList chunks
            const tf_prefill_group far = a.list[chunk];
            start = far.pair_start;
            what = packed(far);
        }
        start = uniform_u32(start);
        what = uniform_u32(what);
        const uint32_t left = (what & 0xFFFFu) - batch * kSliceBatch, count = min(left, kSliceBatch);
        return Unit{chunk, batch, what >> 16, start + batch * kSliceBatch, count, left - count};
    };
    auto unit_after = [&](const Unit &u) {
        if (u.after != 0u) return unit_of(u.chunk, u.batch + 1u);
        uint32_t chunk = u.chunk + 1u;
        Unit next;
        for (; chunk < n_chunks; ++chunk) {
            next = unit_of(chunk, 0u);
            if (next.count != 0u) return next;         // a chunk without pairs is no unit
        }
        return Unit{n_chunks, 0u, 0u, 0u, 0u, 0u};
    };
    if (!placed) {
        auto place_of = [&](uint32_t spent) {
            Place at = {n_chunks, 0u, 0u};
            if (spent >= cost) return at;
            for (uint32_t r = 0; 64u * r < n_chunks; ++r) {
                uint32_t from, what;
                asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(from), "=&v"(what) : "v"(table + 4u * (64u * r + (uint32_t)lane)), "n"(8 * kSliceList) : "memory");
                if (place_among(spent, 64u * r, from, what & 0xFFFFu, at)) break;
            }
            return at;
        };
        first = place_of(share_at(0u));
        last = place_of(share_at(1u));
    }
    if (first.chunk == last.chunk && first.batch == last.batch && first.tile == last.tile) return;

    // ---- requests of weights
    const uint32_t ring = lds + kSliceRing + (uint32_t)wave * 2u * kSliceSlot;
    const uint32_t w_lane = (uint32_t)(lane >> 3) * row_bytes + (uint32_t)g0 * 32u + (uint32_t)((lane & 7) ^ (lane >> 3)) * 16u;
    const int sb_row = lane >> 1, sb_half = (GATE_UP && sb_row >= 16) ? 1 : 0;
    const uint32_t sb_lane = (uint32_t)(GATE_UP ? sb_row & 15 : sb_row) * sb_row_bytes + (uint32_t)g0 * 2u + (uint32_t)(lane & 1) * 4u;
    const uint8_t *const s_lane = (sb_half ? p.s[1] : p.s[0]) + sb_lane, *const b_lane = (sb_half ? p.b[1] : p.b[0]) + sb_lane;
    Unit unit = unit_of(first.chunk, first.batch);
    // the next tile to ask for; tiles asked for so far; whether there is one
    Unit ask_unit = unit;
    uint32_t ask_tile = first.tile, asked = 0u;
    bool to_ask = true;
    auto ask_next = [&] {
        if (!to_ask) return;
        if (working) {
            const uint64_t expert_at = ask_unit.expert * p.stride;
            const uint32_t row0 = min(ask_tile * (uint32_t)p.row_groups + (uint32_t)rg, tiles - 1u) * kRows;     // past the last tile: it again, never stored
            const uint32_t to = ring + (asked & 1u) * kSliceSlot;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint8_t *w = GATE_UP ? p.w[t >> 1] + expert_at + (size_t)(row0 + 8u * (t & 1)) * row_bytes : p.w[0] + expert_at + (size_t)(row0 + 8u * t) * row_bytes;
                slice_copy16(uniform_ptr(w) + w_lane, to + 1024u * t);      // (non-temporal: 2.33 -> 2.5 us a tile)
            }
            const uint64_t sb_at = expert_at + (size_t)row0 * sb_row_bytes;
            slice_copy4(GATE_UP ? s_lane + sb_at : uniform_ptr(p.s[0] + sb_at) + sb_lane, to + kSliceWBytes);
            slice_copy4(GATE_UP ? b_lane + sb_at : uniform_ptr(p.b[0] + sb_at) + sb_lane, to + kSliceWBytes + 256u);
            stay_in_order();
        }
        ++asked;
        if (++ask_tile == positions) {
            ask_unit = unit_after(ask_unit);
            ask_tile = 0u;
        }
        to_ask = !(ask_unit.chunk == last.chunk && ask_unit.batch == last.batch && ask_tile == last.tile);
    };

    const uint32_t w_read = ring + (uint32_t)i * 128u + (uint32_t)(kb ^ (i & 7)) * 16u, sb_read = ring + kSliceWBytes + (uint32_t)i * 8u;
    const uint32_t sums = lds + kSliceSumsAt, own_area = sums + (uint32_t)wave * kSliceSums, own_sums = own_area + (uint32_t)lane * 16u;
    const uint32_t group_sums = sums + (uint32_t)(rg * p.slices) * kSliceSums;

    // The sum over the slices of the four bytes at `from` + the slice's place
    auto over_slices = [&](uint32_t from) {
        float total = 0.0f;
        if (p.row_groups == 1) {                               // seven to twelve slices, requested together (there are twelve places)
            float v[kSliceMaxWaves];
            asm volatile("ds_read_b32 %0, %12\n\tds_read_b32 %1, %12 offset:4096\n\tds_read_b32 %2, %12 offset:8192\n\tds_read_b32 %3, %12 offset:12288\n\t"
                         "ds_read_b32 %4, %12 offset:16384\n\tds_read_b32 %5, %12 offset:20480\n\tds_read_b32 %6, %12 offset:24576\n\tds_read_b32 %7, %12 offset:28672\n\t"
                         "ds_read_b32 %8, %12 offset:32768\n\tds_read_b32 %9, %12 offset:36864\n\tds_read_b32 %10, %12 offset:40960\n\tds_read_b32 %11, %12 offset:45056\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
                         : "v"(from) : "memory");
#pragma unroll
            for (int w = 0; w < kSliceMaxWaves; ++w)
                if (w < 7 || w < p.slices) total += v[w];
        } else {
            for (int w = 0; w < p.slices; w += 3) {
                float v[3];
                asm volatile("ds_read_b32 %0, %3\n\tds_read_b32 %1, %4\n\tds_read_b32 %2, %5\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2])
                             : "v"(from + (uint32_t)w * kSliceSums), "v"(from + (uint32_t)min(w + 1, p.slices - 1) * kSliceSums), "v"(from + (uint32_t)min(w + 2, p.slices - 1) * kSliceSums)
                             : "memory");
                total += v[0];
                if (w + 1 < p.slices) total += v[1];
                if (w + 2 < p.slices) total += v[2];
            }
        }
        return total * 16777216.0f;
    };
    // Adds up the sums of the block's tile number `at`, position `tile_pos` of the unit, and writes the outputs.  `pieces` pieces of sums a wave (8
    // pairs each); with no more than two of them a wave's sums have two places in turn.  The group's waves share them out in parts of 64 outputs, the
    // first ones in turn: one wave at all of a tile's outputs held the others up at the barrier behind (8 / 32 pairs a unit, gate / up, 2.6 / 3.1
    // us a tile; without any adding up 2.1 / 2.5).
    auto reduce = [&](uint32_t first_pair, uint32_t pair_count, uint32_t at, uint32_t tile_pos, uint32_t pieces) {
        if (!working) return;
        const uint32_t out_stride = (uint32_t)p.out_stride;
        const uint32_t set = pieces <= 2u ? (at & 1u) * (kSliceSums / 2) : 0u;
        const uint32_t tile = tile_pos * (uint32_t)p.row_groups + (uint32_t)rg;
        if constexpr (!GATE_UP) {
            // few slices, as a rule: a wave takes a whole piece, four pairs of a row a lane, in one trip to LDS
            for (uint32_t piece = ((uint32_t)slice + at) % (uint32_t)p.slices; piece < pieces; piece += (uint32_t)p.slices) {
                const uint32_t pair = 8u * piece + 4u * (uint32_t)kb, from = group_sums + set + piece * 1024u + (uint32_t)lane * 16u;
                f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                u32x4 row;
                for (int w = 0; w < p.slices; w += 3) {
                    f32x4 q0, q1, q2;
                    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\ts_waitcnt lgkmcnt(0)"
                                 : "=&v"(q0), "=&v"(q1), "=&v"(q2), "=&v"(row)
                                 : "v"(from + (uint32_t)w * kSliceSums), "v"(from + (uint32_t)min(w + 1, p.slices - 1) * kSliceSums),
                                   "v"(from + (uint32_t)min(w + 2, p.slices - 1) * kSliceSums), "v"(lds + kSliceRowsAt + 4u * pair)
                                 : "memory");
                    v += q0;
                    if (w + 1 < p.slices) v += q1;
                    if (w + 2 < p.slices) v += q2;
                }
                if (tile < tiles) {
                    half_t *const o = p.out + (tile * 32u + (uint32_t)i);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (pair + j < pair_count) o[(uint64_t)row[j] * out_stride] = (half_t)(v[j] * 16777216.0f);
                }
            }
        } else {
            const uint32_t parts = 2u * pieces, e = (uint32_t)lane & 3u, c = (uint32_t)lane >> 2;            // of four pairs by sixteen columns
            for (uint32_t part = ((uint32_t)slice + at * parts) % (uint32_t)p.slices; part < parts; part += (uint32_t)p.slices) {
                const uint32_t pair = 4u * part + e, from = group_sums + set + part * 512u + (uint32_t)lane * 4u;      // 16 gate columns, then the same of up
                float gate = over_slices(from), up = over_slices(from + 256u);
                if (shared) {                                                                              // the row chain's stage boundary
                    gate = (float)(half_t)gate;
                    up = (float)(half_t)up;
                }
                if (pair < pair_count && tile < tiles)
                    p.out[(uint64_t)(first_pair + pair - (shared ? 0u : a.pair_base)) * out_stride + (tile * 16u + c)] = (half_t)(gelu_tanh_fast(gate) * up);
            }
        }
    };

    // The unit's pairs, 16 bytes each, into LDS: word by word, they are aligned to four bytes; past the last the last again
    auto copy_pairs = [&](const Unit &u, uint32_t to) {
        uint32_t l = (uint32_t)lane;
        asm volatile("" : "+v"(l));                            // addresses are made here, no registers keep them
#pragma unroll
        for (uint32_t h = 0; h < 2u; ++h)
            slice_copy4(reinterpret_cast<const uint32_t *>(a.pairs + (u.first + min(16u * h + (l >> 2), u.count - 1u))) + (l & 3u), to + 256u * h);
    };
    // the unit before: its pairs, its last tile; done: tiles behind this block
    uint32_t before_first = 0u, before_pairs = 0u, before_tile = 0u, before_pieces = 0u, before_count = 0u, done = 0u;
    for (uint32_t tile0 = first.tile;; tile0 = 0u) {
        const bool closing = unit.chunk == last.chunk && unit.batch == last.batch;
        const uint32_t count = (closing ? last.tile : positions) - tile0;
        // The unit's pairs: the first unit's behind each wave's second tile, ahead of the first weights; a later unit's have been put into
        // LDS while the unit before was worked on.
        uint32_t pairs_at = lds + kSlicePairsAt;
        if (done == 0u) {
            pairs_at = ring + kSliceSlot + kSliceWBytes;
            if (!shared) copy_pairs(unit, pairs_at);
            stay_in_order();
            ask_next();
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kSliceCopies) : "memory");
        } else {
            reduce(before_first, before_pairs, done - 1u, before_tile, before_pieces);
            if (wave == 0 && before_count < 3u) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the pairs: no tile's wait has covered them
            slice_barrier();                                   // the sums and rows of the unit before are done with, the pairs are there
        }
        if constexpr (!GATE_UP) {
            if (wave == 0 && lane < 32) {
                uint32_t row = unit.first + (uint32_t)i;       // of a shared expert: its own
                if (!shared) {
                    u32x4 pair;
                    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(pair) : "v"(pairs_at + 16u * (uint32_t)i) : "memory");
                    row = pair[0] * a.top_k + pair[2];         // token * top_k + rank
                }
                lds_put4(lds + kSliceRowsAt + 4u * (uint32_t)i, row);
            }
        }
        // The activations come through LDS, eight rows of 512 bytes at a time, whole lines (a load of "its" 16 bytes of its own row by each
        // lane is a look-up a lane: 5 us for the sixteen of every wave): into the wave's sums, and where there are more than eight rows, into the
        // tile that has not been asked for.  Piece p of row r sits at p ^ (r & 7).
        const uint32_t free_tile = ring + (asked & 1u) * kSliceSlot;
        auto fetch = [&](uint32_t first_row, uint32_t to) {
            uint32_t rows[4], source[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) rows[j] = min(first_row + 2u * j + (uint32_t)kb, unit.count - 1u);
            if (GATE_UP && !shared) {
                asm volatile("ds_read_b32 %0, %4\n\tds_read_b32 %1, %5\n\tds_read_b32 %2, %6\n\tds_read_b32 %3, %7\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(source[0]), "=&v"(source[1]), "=&v"(source[2]), "=&v"(source[3])
                             : "v"(pairs_at + 16u * rows[0]), "v"(pairs_at + 16u * rows[1]), "v"(pairs_at + 16u * rows[2]), "v"(pairs_at + 16u * rows[3])
                             : "memory");
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) source[j] = unit.first + rows[j] - (shared ? 0u : a.pair_base);
            }
            if (working) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (first_row + 2u * j < unit.count)
                        slice_copy16(p.x + ((size_t)source[j] * (size_t)p.x_stride + (uint32_t)g0 * 64u + (uint32_t)(i ^ (2 * j + kb)) * 8u), to + 1024u * j);
            }
            stay_in_order();
        };
        u32x4 raw[kSliceGroups][4] = {};
        auto take = [&] {
            const uint32_t x_at = ((i & 8) ? free_tile : own_area) + (uint32_t)(i & 7) * 512u + (uint32_t)((kb * 4) ^ (i & 7)) * 16u;
            asm volatile("ds_read_b128 %0, %16\n\tds_read_b128 %1, %16 offset:128\n\tds_read_b128 %2, %16 offset:256\n\tds_read_b128 %3, %16 offset:384\n\t"
                         "ds_read_b128 %4, %17\n\tds_read_b128 %5, %17 offset:128\n\tds_read_b128 %6, %17 offset:256\n\tds_read_b128 %7, %17 offset:384\n\t"
                         "ds_read_b128 %8, %18\n\tds_read_b128 %9, %18 offset:128\n\tds_read_b128 %10, %18 offset:256\n\tds_read_b128 %11, %18 offset:384\n\t"
                         "ds_read_b128 %12, %19\n\tds_read_b128 %13, %19 offset:128\n\tds_read_b128 %14, %19 offset:256\n\tds_read_b128 %15, %19 offset:384\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=&v"(raw[0][0]), "=&v"(raw[1][0]), "=&v"(raw[2][0]), "=&v"(raw[3][0]), "=&v"(raw[0][1]), "=&v"(raw[1][1]), "=&v"(raw[2][1]), "=&v"(raw[3][1]),
                           "=&v"(raw[0][2]), "=&v"(raw[1][2]), "=&v"(raw[2][2]), "=&v"(raw[3][2]), "=&v"(raw[0][3]), "=&v"(raw[1][3]), "=&v"(raw[2][3]), "=&v"(raw[3][3])
                         : "v"(x_at), "v"(x_at ^ 16u), "v"(x_at ^ 32u), "v"(x_at ^ 48u)
                         : "memory");
        };
        const bool early = unit.count <= 8u && to_ask;         // the tile stays free: its weights right behind the activations
        for (uint32_t row0 = 0; row0 < unit.count; row0 += 16u) {
            fetch(row0, own_area);
            if (row0 + 8u < unit.count) fetch(row0 + 8u, free_tile);
            if (early) {
                ask_next();
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kSliceCopies) : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            if (row0 == 0u || i >= 16) take();                 // lanes past the rows there are take whatever is there: sums of pairs that do not exist
        }
        if (!early) ask_next();
        half8_t x[kSliceGroups][4];
        bf16x8_t xs;
        bool lane_odd = false;
        {
            uint32_t part[3][kSliceGroups];
#pragma unroll
            for (int g = 0; g < kSliceGroups; ++g) {
                // a group's 32 values of this lane in the order the nibble masks give: (0, 4), (1, 5), (2, 6), (3, 7) of every eight
                const bool mine = g >= skip;
                float16_t total;
#pragma unroll
                for (int r = 0; r < 16; ++r) total[r] = 0.0f;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const u32x4 v = mine ? raw[g][d] : u32x4{0u, 0u, 0u, 0u};
                    x[g][d] = __builtin_bit_cast(half8_t, u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                                                                __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)});
                    // the sum of all 64 values of the lane's pair: the values as they came against ones, the same in all sixteen rows
                    const half_t one = (half_t)1.0f;
                    total = __builtin_amdgcn_mfma_f32_32x32x16_f16(half8_t{one, one, one, one, one, one, one, one}, __builtin_bit_cast(half8_t, v), total, 0, 0, 0);
                }
                lane_odd = lane_odd || !(fabsf(total[0]) < INFINITY);          // of 64 fp16 numbers: an infinity or NaN is among them
                float rest = total[0] * 5.9604644775390625e-8f;                // in units of 2^24, as the products come out
#pragma unroll
                for (int p = 0; p < 3; ++p) {                                   // eight bits each
                    part[p][g] = __float_as_uint(rest) & 0xFFFF0000u;
                    rest -= __uint_as_float(part[p][g]);
                }
            }
            u32x4 v;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t p0 = part[0][2 * j] >> 16 | part[0][2 * j + 1], p1 = part[1][2 * j] >> 16 | part[1][2 * j + 1], p2 = part[2][2 * j] >> 16 | part[2][2 * j + 1];
                v[j] = lane_odd ? 0u : kb ? p2 : p0;
                v[2 + j] = lane_odd || kb ? 0u : p1;
            }
            xs = __builtin_bit_cast(bf16x8_t, v);
        }

        // the tiles of the unit
        const uint32_t pieces = unit.count <= 8u ? 1u : unit.count <= 16u ? 2u : 4u;
        // (beyond the unit's pairs, and in waves without a slice, the registers hold anything)
        const uint32_t kind = working && ((uint32_t)__ballot(lane_odd) & (0xFFFFFFFFu >> (kSliceBatch - unit.count))) != 0u ? 0u : pieces;
        for (uint32_t t = 0; t < count; ++t) {
            const uint32_t at = done + t;
            // this tile's requests have landed; the next one's, if it has been asked for, may still be on their way.  What a wave
            // stores it stores before it asks again, so nothing else is younger (but for the next unit's pairs, once: then the wait is for more).
            if (asked > at + 1u) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kSliceCopies) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            u32x4 w[kSliceGroups];
            u32x2 s, b;
            {
                const uint32_t wr = w_read + (at & 1u) * kSliceSlot, sr = sb_read + (at & 1u) * kSliceSlot;
                asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\tds_read_b128 %2, %8\n\tds_read_b128 %3, %9\n\tds_read_b64 %4, %10\n\t"
                             "ds_read_b64 %5, %10 offset:256\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(s), "=&v"(b)
                             : "v"(wr), "v"(wr ^ 32u), "v"(wr ^ 64u), "v"(wr ^ 96u), "v"(sr)
                             : "memory");
            }
            if (t > 0) reduce(unit.first, unit.count, at - 1u, tile0 + t - 1u, pieces);
            if (t + 1u < count) ask_next();                                     // the last tile's turn comes behind the next unit's activations
            float16_t acc;
            if (kind == 1u) slice_multiply<SD, 4, false>(x, xs, w, s, b, false, acc);
            else if (kind == 2u) slice_multiply<SD, 8, false>(x, xs, w, s, b, false, acc);
            else if (__builtin_expect(kind != 0u, 1)) slice_multiply<SD, 16, false>(x, xs, w, s, b, false, acc);
            else slice_multiply<SD, 16, true>(x, xs, w, s, b, lane_odd, acc);
            const uint32_t to = own_sums + (pieces <= 2u ? (at & 1u) * (kSliceSums / 2) : 0u);
            if (pieces > 2u) __builtin_amdgcn_s_barrier();                      // the tile before has been added up
            lds_put16(to, f32x4{acc[0], acc[1], acc[2], acc[3]});
            if (pieces > 1u) lds_put16(to + 1024u, f32x4{acc[4], acc[5], acc[6], acc[7]});
            if (pieces > 2u) {
                lds_put16(to + 2048u, f32x4{acc[8], acc[9], acc[10], acc[11]});
                lds_put16(to + 3072u, f32x4{acc[12], acc[13], acc[14], acc[15]});
            }
            slice_barrier();
            // every wave has seen this unit's pairs: the next unit's may take their place (landed by the wait of the second tile from here)
            if (t == 0u && wave == 0 && !closing && !shared) {
                const Unit next = unit_after(unit);
                if (next.count != 0u) copy_pairs(next, lds + kSlicePairsAt);
                stay_in_order();
            }
        }
        before_pieces = pieces;
        before_first = unit.first;
        before_pairs = unit.count;
        before_tile = tile0 + count - 1u;
        before_count = count;
        done += count;
        // done where the share ends, inside this unit or exactly behind it
        if (closing) break;
        unit = unit_after(unit);
        if (unit.chunk == last.chunk && unit.batch == last.batch && last.tile == 0u) break;
    }
    reduce(before_first, before_pairs, done - 1u, before_tile, before_pieces);
}

// Token rows of fewer columns have so few slices that adding up weighs more than it saves (d 1024, f 512, 128 experts, 64 / 128 / 300 tokens: quad or
// tiles 45 / 42 / 51 us, slice 39 / 44 / 57; d 1536, f 768: 73 / 68 / 91 and 58 / 66 / 88).  At the line, d 1280, f 640, 128 / 64 experts of 96 tokens, routed 63/56, 41/40
// and with a shared expert of 1280 67/61, 48/44, popular 43/38, 42/37; the shared expert alone 32/22.
constexpr int kSliceMinCols = 1280;
bool slice_width_ok(int k) { return k >= 64 * kSliceGroups && (k >> 6) <= kSliceGroups * kSliceMaxWaves; }
SliceProblem slice_problem(const uint8_t *w0, const uint8_t *s0, const uint8_t *b0, const uint8_t *w1, const uint8_t *s1, const uint8_t *b1, uint64_t stride,
                           const half_t *x, long x_stride, half_t *out, long out_stride, int k, int n) {
    const int slices = ((k >> 6) + kSliceGroups - 1) / kSliceGroups;
    return SliceProblem{{w0, w1}, {s0, s1}, {b0, b1}, stride, x, x_stride, out, out_stride, k, n, slices, kSliceMaxWaves / slices};
}
template <bool GATE_UP>
void launch_slice(tf_ctx *ctx, hipStream_t st, const SliceArgs &a, tf_dtype sd) {
    // as many waves as the problems use: twelve, or fewer where their slices leave a remainder
    const int waves = std::max(a.list_cap ? a.routed.slices * a.routed.row_groups : 0, a.shared_rows ? a.shared.slices * a.shared.row_groups : 0);
    const dim3 grid((uint32_t)ctx->num_cus), block((uint32_t)(64 * waves));
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, a); };
    if (a.list_cap > kSliceList) sd == TF_BF16 ? launch(grouped_slice_kernel<GATE_UP, 0, true>) : launch(grouped_slice_kernel<GATE_UP, 1, true>);
    else sd == TF_BF16 ? launch(grouped_slice_kernel<GATE_UP, 0, false>) : launch(grouped_slice_kernel<GATE_UP, 1, false>);
}

}  // namespace

namespace tfk {

bool grouped_slice_ok(const ExpertTable &tab, const ChunkList &cl, uint32_t pair_count, int d, int f) {
    return tab.pool != nullptr && cl.dev != nullptr && pair_count != 0 && pair_count < 65536 && tab.num_experts <= 65536 &&
           d >= kSliceMinCols && slice_width_ok(d) && slice_width_ok(f);
}

// gate / up / GeGLU of a shared expert's rows, and its down product
static SliceProblem shared_gate_up(const DenseRide &r) {
    const uint8_t *w[2] = {at(r.gate->weights, r.gate->weights_offset), at(r.up->weights, r.up->weights_offset)};
    const uint8_t *s[2] = {at(r.gate->scales, r.gate->scales_offset), at(r.up->scales, r.up->scales_offset)};
    const uint8_t *b[2] = {at(r.gate->biases, r.gate->biases_offset), at(r.up->biases, r.up->biases_offset)};
    return slice_problem(w[0], s[0], b[0], w[1], s[1], b[1], 0, r.x, r.ldx, r.acts, (long)r.gate->rows, (int)r.gate->cols, (int)r.gate->rows);
}
static SliceProblem shared_down(const DenseRide &r) {
    const uint8_t *w = at(r.down->weights, r.down->weights_offset), *s = at(r.down->scales, r.down->scales_offset), *b = at(r.down->biases, r.down->biases_offset);
    return slice_problem(w, s, b, w, s, b, 0, r.acts, (long)r.down->cols, r.y, r.ldy, (int)r.down->cols, (int)r.down->rows);
}

bool shared_slice_ok(const tf_projection *gate) { return (int)gate->cols >= kSliceMinCols && slice_width_ok((int)gate->cols) && slice_width_ok((int)gate->rows); }

int32_t launch_shared_slice(tf_ctx *ctx, hipStream_t st, const DenseRide &ride, tf_dtype sd) {
    SliceArgs a = {};
    a.shared_rows = (uint32_t)ride.rows;
    a.shared = shared_gate_up(ride);
    launch_slice<true>(ctx, st, a, sd);
    const int32_t rc = check_launch(ctx, "shared expert gate / up slice");
    if (rc != TF_OK) return rc;
    a.shared = shared_down(ride);
    launch_slice<false>(ctx, st, a, sd);
    return check_launch(ctx, "shared expert down slice");
}

int32_t launch_grouped_slice(tf_ctx *ctx, hipStream_t st, const ExpertTable &tab, const tf_expert_offsets &off, const ChunkList &cl,
                             uint32_t n_chunks_upper, const GroupedGeom &g, tf_dtype sd, const DenseRide *ride) {
    SliceArgs a = {};
    a.list = cl.dev;
    a.list_count = cl.dev_n;
    a.list_cap = n_chunks_upper;
    a.num_experts = tab.num_experts;
    a.pairs = g.pairs;
    a.pair_base = g.acts_pair_base;
    a.top_k = (uint32_t)g.top_k;
    const uint8_t *pool = tab.pool;
    a.routed = slice_problem(pool + off.gate_W_off, pool + off.gate_s_off, pool + off.gate_b_off, pool + off.up_W_off, pool + off.up_s_off, pool + off.up_b_off,
                             tab.stride, g.hidden, g.hidden_stride, g.acts, g.f, g.d, g.f);
    if (ride) {
        a.shared_rows = (uint32_t)ride->rows;
        a.shared = shared_gate_up(*ride);
    }
    launch_slice<true>(ctx, st, a, sd);
    const int32_t rc = check_launch(ctx, "grouped phase 1 slice");
    if (rc != TF_OK) return rc;
    const uint8_t *w = pool + off.down_W_off, *s = pool + off.down_s_off, *b = pool + off.down_b_off;
    a.routed = slice_problem(w, s, b, w, s, b, tab.stride, g.acts, g.f, g.route_partials, g.d, g.f, g.d);
    if (ride) a.shared = shared_down(*ride);
    launch_slice<false>(ctx, st, a, sd);
    return check_launch(ctx, "grouped down slice");
}

}  // namespace tfk
