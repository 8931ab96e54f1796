// isp_linear_rows_f32: fp32 products of any number of rows.  Which tile one takes, its launch (the kernel: linear_tiled_f32.h) and the
// addition of split sums.
// The library's kernels (hipBLASLt) do these at 78 to 98 TFLOP/s for a few hundred rows and read the weights of a few at 1.7 to 4.4
// TB/s.  us before and after, addition of splits included: 308 rows x 2048 -> 6144 79, 63; x 2048 -> 2048 33, 28; x 2048 -> 11264 174,
// 119; x 5632 -> 2048 74, 60; 16 x 4096 -> 12288 46, 37; 64 x 11008 -> 4096 105, 53.  Over 250 products of models of 512 ... 5120
// columns, 1 ... 3000 rows: 1.43 times as fast in the geometric mean, 0.89 times at worst (668 x 9792 -> 2560, whose tiles fill the chip
// badly).  Whole layers of 3000 to 16000 rows x 4096 to 6144 take 0.90 to 1.025 times what they do with the library's products, longest where
// rows are a multiple of 2048 (8192 x 4096, inter 11008: 24.1 ms, 23.5 with the library's; 8000 rows 23.7, 23.7).  The matrix cores' fp32 rate bounds all but few rows: 116 to 147 of 157 TFLOP/s.
#include "linear_tiled_f32.h"

#include <math.h>

#include "linear_rows.h"

namespace isp {

// A tile and what it measured: a workgroup takes start_us, and per 32 k what is longer of lone_us (a compute unit to itself) and of
// shared_us times the workgroups of its compute unit, up to per_unit; weights arrive at stream_tb TB/s at most and sums leave at
// sums_tb.  Fitted (mean error 3 to 5 %) to 5900 timings of 250 products, each with every tile and up to sixteen splits.  The plan
// that these figures choose is 2 % behind the best of all (geometric mean; 10 % in one of twenty).
struct TiledTileF32 {
    int rows, cols, per_unit;
    float start_us, lone_us, shared_us, stream_tb, sums_tb;
};
constexpr TiledTileF32 kTilesF32[] = {
    {32, 64, 3, 3.24f, 0.232f, 0.240f, 6.33f, 8.90f}, {32, 128, 2, 3.19f, 0.454f, 0.466f, 6.03f, 6.90f},
    {64, 128, 2, 2.92f, 0.917f, 0.888f, 5.10f, 5.67f}, {96, 64, 2, 2.61f, 0.700f, 0.675f, 4.13f, 5.77f},
    {160, 64, 2, 3.18f, 1.128f, 1.088f, 2.54f, 6.30f},
};

TiledPlan tiled_plan_f32(int m, int n, int k, int max_splits, double* us_of_plan) {
    const int steps = (k + kTiledStepF32 - 1) / kTiledStepF32, units = resident_waves() / 32;
    const double mn = (double)m * n, weight_bytes = 4.0 * n * k;
    TiledPlan best = {0, 1, steps};
    double best_us = 0.0;
    for (int c = 0; c < (int)(sizeof(kTilesF32) / sizeof(kTilesF32[0])); c++) {
        const TiledTileF32& tile = kTilesF32[c];
        if (tile.rows >= 2 * m && tile.rows > 32) continue;  // rows of a tile that do not exist are work for nothing
        const long long tiles = ((m + tile.rows - 1ll) / tile.rows) * ((n + tile.cols - 1) / tile.cols), slots = (long long)units * tile.per_unit;
        const double stream = 2.0 + weight_bytes / tile.stream_tb * 1e-6;
        for (int s = 1; s <= max_splits && (s == 1 || (2 * s <= steps && tiles * (s - 1) < slots)); s++) {
            const int per = (steps + s - 1) / s;
            if (s > 1 && per * (s - 1) >= steps) continue;  // the same as a smaller number
            const long long groups = tiles * s, whole = groups / slots, rest = groups - whole * slots;
            const auto round = [&](int sharing) {
                const double step = tile.shared_us * sharing;
                return sharing == 0 ? 0.0 : tile.start_us + per * (step > tile.lone_us ? step : (double)tile.lone_us);
            };
            double us = (double)whole * round(tile.per_unit) + round((int)((rest + units - 1) / units));
            // partial sums: written here in place of the product; the kernel that adds them takes 2.5 us and 4.5 TB/s
            const double sums = s == 1 ? 0.0 : 4.0 * (s - 1) * mn / tile.sums_tb * 1e-6 + 2.5 + 4.0 * (s + 1) * mn / 4.5 * 1e-6;
            us = sqrt(sqrt(us * us * us * us + stream * stream * stream * stream)) + sums;
            if (best_us == 0.0 || us < best_us) {
                best_us = us;
                best = {c, s, per};
            }
        }
    }
    if (us_of_plan) *us_of_plan = best_us;
    return best;
}

// out = sum over the splits, in their order; four columns per lane.
__global__ __launch_bounds__(kBlock) void linear_add_splits_f32(const float* __restrict__ partial, float* __restrict__ out,
                                                                unsigned quads, int splits) {
    const unsigned i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= quads) return;
    const float* const at[1] = {partial + 4 * (size_t)i};
    float4v sum[1];
    add_splits(at, 4 * (size_t)quads, splits, sum);
    reinterpret_cast<float4v*>(out)[i] = sum[0];
}

// Extents that the kernels can count (the addition indexes four values in 32 bits).
static bool linear_shape_f32(int m, int n, int k) {
    return k > 0 && n % 4 == 0 && k % 4 == 0 && n <= kTiledMaxExtent && k <= kTiledMaxExtent && m <= kTiledMaxRowsF32 &&
           (long long)m * n < kTiledMaxValues;
}

template <bool SWIGLU>
static void launch_f32(const TiledPlan& plan, const float* a, const float* w, float* out, int m, int n, int k, hipStream_t stream) {
    const TiledTileF32& tile = kTilesF32[plan.tile];
    const int cols = SWIGLU ? tile.cols / 2 : tile.cols, width = SWIGLU ? n / 2 : n;
    const dim3 grid((unsigned)((m + tile.rows - 1ll) / tile.rows) * (unsigned)((width + cols - 1) / cols), (unsigned)plan.splits);
#define ISP_TILED(INDEX, BM, BN, WM, WN, STAGES)                                                                              \
    case INDEX:                                                                                                               \
        static_assert(kTilesF32[INDEX].rows == BM && kTilesF32[INDEX].cols == BN, "tile");                                    \
        hipLaunchKernelGGL((linear_tiled_f32<BM, BN, WM, WN, STAGES, SWIGLU>), grid, dim3(kWave * WM * WN), 0, stream, a, w, out, m,  \
                           n, k, plan.steps_per_split);                                                                       \
        break
    switch (plan.tile) {
        ISP_TILED(0, 32, 64, 2, 2, 4);
        ISP_TILED(1, 32, 128, 1, 4, 4);
        ISP_TILED(2, 64, 128, 2, 2, 3);
        ISP_TILED(3, 96, 64, 2, 2, 3);
        ISP_TILED(4, 160, 64, 2, 2, 2);
    }
#undef ISP_TILED
}

void launch_tiled_f32(const TiledPlan& plan, const float* a, const float* w, float* out_or_partial, int m, int n, int k, hipStream_t stream) {
    launch_f32<false>(plan, a, w, out_or_partial, m, n, k, stream);
}

void launch_tiled_swiglu_f32(const TiledPlan& plan, const float* a, const float* gate_up, float* out, int m, int inter, int k,
                             hipStream_t stream) {
    launch_f32<true>(plan, a, gate_up, out, m, 2 * inter, k, stream);
}

static int linear_f32(const float* a, const float* w, float* out, float* workspace, int m, int n, int k, hipStream_t stream) {
    if (m < 0 || n < 0 || k < 0) return ISP_ERR_BAD_SHAPE;
    if (m == 0 || n == 0) return ISP_OK;
    if (!linear_shape_f32(m, n, k)) return ISP_ERR_UNSUPPORTED;
    ISP_REQUIRE_PTR(a);
    ISP_REQUIRE_PTR(w);
    ISP_REQUIRE_PTR(out);
    if (!aligned16(a) || !aligned16(w) || !aligned16(out)) return ISP_ERR_UNSUPPORTED;
    const TiledPlan plan = tiled_plan_f32(m, n, k, kTiledMaxSplits, nullptr);
    if (plan.splits > 1) {
        ISP_REQUIRE_PTR(workspace);
        if (!aligned16(workspace)) return ISP_ERR_UNSUPPORTED;
    }
    launch_f32<false>(plan, a, w, plan.splits > 1 ? workspace : out, m, n, k, stream);
    const int status = note_launch(hipGetLastError());
    if (status != ISP_OK || plan.splits == 1) return status;
    const unsigned quads = (unsigned)((size_t)m * (size_t)n / 4);
    hipLaunchKernelGGL(linear_add_splits_f32, dim3((quads + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, workspace, out, quads,
                       plan.splits);
    return note_launch(hipGetLastError());
}

}  // namespace isp

extern "C" {

size_t isp_linear_rows_f32_workspace(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || !isp::linear_shape_f32(m, n, k)) return 0;
    const isp::TiledPlan plan = isp::tiled_plan_f32(m, n, k, isp::kTiledMaxSplits, nullptr);
    return plan.splits == 1 ? 0 : (size_t)plan.splits * (size_t)m * (size_t)n * sizeof(float);
}

int isp_linear_rows_f32(const void* a, const void* w, void* out, void* workspace, int m, int n, int k, isp_stream_t stream) {
    return isp::linear_f32(static_cast<const float*>(a), static_cast<const float*>(w), static_cast<float*>(out),
                           static_cast<float*>(workspace), m, n, k, static_cast<hipStream_t>(stream));
}

int isp_linear_rows_f32_plan(int m, int n, int k, int* tile_rows, int* tile_cols, int* splits) {
    if (m <= 0 || n <= 0 || k <= 0 || !isp::linear_shape_f32(m, n, k)) return ISP_ERR_BAD_SHAPE;
    ISP_REQUIRE_PTR(tile_rows);
    ISP_REQUIRE_PTR(tile_cols);
    ISP_REQUIRE_PTR(splits);
    const isp::TiledPlan plan = isp::tiled_plan_f32(m, n, k, isp::kTiledMaxSplits, nullptr);
    *tile_rows = isp::kTilesF32[plan.tile].rows;
    *tile_cols = isp::kTilesF32[plan.tile].cols;
    *splits = plan.splits;
    return ISP_OK;
}

}  // extern "C"
