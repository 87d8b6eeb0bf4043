// Launches of the split kernels (tf_qmm_split.hpp) and the rules that choose between them.
#include "tf_qmm_split.hpp"

using namespace tfk;

namespace {

template <int BITS, int SD, int MT, int NJ, int NW, int GP, bool GEGLU>
__global__ __launch_bounds__(64 * NW) void qmm_split_kernel(SplitArgs a) {
    __shared__ __align__(128) uint8_t lds[SplitGeom<BITS, MT, NJ, NW, GP>::kLds];
    qmm_split_body<BITS, SD, MT, NJ, NW, GP, GEGLU>(a, blockIdx.x, lds);
}

template <int BITS, int MT, int NJ, int NW, int GP, bool GEGLU>
void launch_split(hipStream_t st, const SplitArgs &a, tf_dtype sd) {
    constexpr int cols = GEGLU ? 32 : 32 * NJ;
    const dim3 grid((uint32_t)((a.N + cols - 1) / cols) * (uint32_t)((a.M + 32 * MT - 1) / (32 * MT)));
    if (sd == TF_BF16) hipLaunchKernelGGL((qmm_split_kernel<BITS, 0, MT, NJ, NW, GP, GEGLU>), grid, dim3(64 * NW), 0, st, a);
    else hipLaunchKernelGGL((qmm_split_kernel<BITS, 1, MT, NJ, NW, GP, GEGLU>), grid, dim3(64 * NW), 0, st, a);
}

}  // namespace

namespace tfk {

// Which kernel for M x N x K, in microseconds for the shapes below (K = 2816, weights from HBM; `tiles`: the 128 x 256 tile kernel; the
// others by rows x columns of a block's tile).  A block has a CU to itself, so what counts is how often the device's CUs (here 256) are filled:
//     rows x columns    32 x 32   64 x 32   64 x 64    tiles
//        53 x 2048         8.0      10.2      14.1      26.9
//       128 x 2048         8.7      10.4      14.4      33.9
//       128 x 4096        15.7      11.7      15.7      34.8
//       256 x 4096        27.6      20.1      16.0      34.7
//       500 x 4096        53.9      37.2      28.6      35.5
//       500 x 8192         107      72.6      53.4      37.2
// So: the smallest tile that fits the chip in one go; 64 x 64 in two goes while the tile kernel would multiply full row tiles (up to
// 64 rows it takes 27 - 29 us, no more than two goes do).  Other contractions, 1 to 1200 rows of 64 to 8192 columns against the tile kernel alone:
// K 8192 1.0 to 4 times as fast (53 x 2816 70.8 -> 17.6 us, 500 x 2816 in two goes 94.1 -> 63.6), K 1024 1.1 to 2.2 times in one go
// but no gain in two (500 x 4096 16.8 -> 17.6 us; a thousand more of K are 6.3 us in two goes and 10.4 on the tiles).  Contractions shorter than a pair of groups a wave, or longer than the waves'
// scale areas hold, stay with the tile kernel.
constexpr int kTwoGoesK = 1280;
int qmm_split_variant(int m, int n, int k, long ldx, int num_cus) {
    if (k < 1024 || k > 8192 || ldx > (1l << 24)) return kSplitNone;
    const int64_t cus = num_cus;
    auto blocks = [&](int rows, int cols) { return (int64_t)((m + (int64_t)rows - 1) / rows) * ((n + (int64_t)cols - 1) / cols); };
    if (blocks(32, 32) <= cus) return kSplit32x32;
    if (blocks(64, 32) <= cus) return kSplit64x32;
    if (blocks(64, 64) <= (m > 64 && k >= kTwoGoesK ? 2 * cus : cus)) return kSplit64x64;
    return kSplitNone;
}

int32_t launch_qmm_split(tf_ctx *ctx, hipStream_t st, int variant, const uint8_t *w, const uint8_t *s, const uint8_t *b, const half_t *x, long ldx,
                         half_t *y, long ldy, int m, int n, int k, tf_dtype sd) {
    const SplitArgs a = qmm_split_args(w, s, b, x, ldx, y, ldy, m, n, k);
    const bool wide = k > 4096;       // twice the scales to keep
    if (variant == kSplit32x32) {
        if (wide) launch_split<4, 1, 1, 8, 8, false>(st, a, sd);
        else launch_split<4, 1, 1, 8, 4, false>(st, a, sd);
    } else if (variant == kSplit64x32) {
        if (wide) launch_split<4, 2, 1, 4, 16, false>(st, a, sd);
        else launch_split<4, 2, 1, 4, 8, false>(st, a, sd);
    } else {
        if (wide) launch_split<4, 2, 2, 4, 16, false>(st, a, sd);
        else launch_split<4, 2, 2, 4, 8, false>(st, a, sd);
    }
    return check_launch(ctx, "int4_qmm");
}

bool geglu_split_ok(const tf_projection *gate, long ldx) { return gate->cols <= 4096 && gate->rows <= 4096 && ldx <= (1l << 24); }

int32_t launch_geglu_split(tf_ctx *ctx, hipStream_t st, const tf_projection *gate, const tf_projection *up, const half_t *x, long ldx, half_t *a_out,
                           long lda, int m, tf_dtype sd) {
    launch_split<4, 1, 2, 8, 4, true>(st, geglu_split_args(gate, up, x, ldx, a_out, lda, m), sd);
    return check_launch(ctx, "prefill_shared_expert gate/up");
}

// The 8-bit shared expert of a block of rows (what a wave keeps of scales ends at 4096 columns).
bool shared8_split_ok(const tf_projection *gate, long ldx) { return gate->cols <= 4096 && gate->rows <= 4096 && ldx <= (1l << 24); }

int32_t launch_shared8_split(tf_ctx *ctx, hipStream_t st, const tf_projection *gate, const tf_projection *up, const tf_projection *down, const half_t *x,
                             long ldx, half_t *acts, half_t *y, long ldy, int m, tf_dtype sd) {
    const int f = (int)gate->rows, d = (int)gate->cols;
    auto blocks = [&](int n, int rows, int cols) { return (int64_t)((m + (int64_t)rows - 1) / rows) * ((n + (int64_t)cols - 1) / cols); };
    const SplitArgs a1 = geglu_split_args(gate, up, x, ldx, acts, (long)f, m);
    if (blocks(f, 32, 32) <= ctx->num_cus) launch_split<8, 1, 2, 4, 8, true>(st, a1, sd);
    else launch_split<8, 2, 2, 4, 8, true>(st, a1, sd);
    const uint8_t *w = at(down->weights, down->weights_offset), *s = at(down->scales, down->scales_offset), *b = at(down->biases, down->biases_offset);
    const SplitArgs a2 = qmm_split_args(w, s, b, acts, (long)f, y, ldy, m, d, f);
    if (blocks(d, 32, 32) <= ctx->num_cus) launch_split<8, 1, 1, 8, 4, false>(st, a2, sd);
    else if (blocks(d, 64, 32) <= ctx->num_cus) launch_split<8, 2, 1, 4, 8, false>(st, a2, sd);
    else launch_split<8, 2, 2, 4, 8, false>(st, a2, sd);
    return check_launch(ctx, "shared expert 8-bit block");
}

}  // namespace tfk
