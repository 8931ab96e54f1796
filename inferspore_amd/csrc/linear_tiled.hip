// Which tile a product of many rows takes, and its launch (the kernel: linear_tiled.h).
#include "linear_rows.h"
#include "linear_tiled.h"

#include <math.h>

namespace isp {

// A tile and what it measured: a workgroup takes start_us + step_us per 64 k with a compute unit to itself, pair_us per 64 k where two
// share one (tiles of up to 80 KiB of LDS); the weights arrive at stream_tb TB/s at most.  Fitted (mean error 7 to 9 %) to 1970
// products of 17 ... 8192 rows over the layers of models of 512 ... 5120 columns, each with every tile and up to sixteen splits; then two
// prices were corrected by measurement.
// swiglu: steps of a product with SwiGLU inside take so much longer.  The wavefronts of 128 x 192 own 96 columns, in which gates and up
// projections alternate 32 bytes at a time, not 64: 1.34 to 1.69 us per step and pair, not 1.22.  Without the factor 660 x 4096 x 22016 took
// 173 us there (128 x 256: 152), 463 rows 104 (256 x 256: 100), 300 rows 93 (192 x 256: 86).  The 192 x 256 tile's step is not the
// fit's 1.166: at 200 to 256 workgroups, for which it is mostly taken, it measures 1.21 to 1.26 (2611 x 4096 x 4096 87.1 us, 128 x 192 82.8;
// x 11008 x 4096 219.6 and 213.1).
// With these figures the plan is 3 % behind the best tile and splits for each of 398 other products of 65 to 8192 rows (geometric mean; 17 %
// in one of twenty).  Worst are 90 to 140 rows and more than 22000 columns: 112 x 5120 x 26176 takes 64 x 128, 74 us, where 128 x 128
// takes 55.  Against the library, of 166 products that take it more than 30 us: 1.29 times as fast in the geometric mean, 0.79 times at
// worst (the same product), slower for 16 of them.
struct TiledTile {
    int rows, cols, threads, per_unit;
    float start_us, step_us, pair_us, stream_tb, partial_tb, swiglu;
};
constexpr TiledTile kTiles[] = {
    {256, 256, 512, 1, 8.38f, 1.301f, 0.0f, 3.62f, 7.59f, 1.0f}, {192, 256, 512, 1, 6.67f, 1.21f, 0.0f, 3.51f, 7.83f, 1.0f},
    {256, 128, 512, 1, 5.16f, 0.731f, 0.0f, 3.41f, 5.88f, 1.0f}, {128, 256, 512, 1, 5.65f, 0.757f, 0.0f, 3.63f, 6.50f, 1.0f},
    {128, 192, 256, 2, 4.01f, 0.887f, 1.216f, 4.09f, 5.10f, 1.25f}, {128, 128, 512, 1, 3.65f, 0.493f, 0.0f, 3.46f, 5.76f, 1.0f},
    {128, 64, 256, 2, 2.21f, 0.382f, 0.645f, 3.59f, 5.15f, 1.0f}, {64, 128, 256, 2, 2.43f, 0.430f, 0.730f, 4.89f, 5.40f, 1.0f},
    {64, 64, 256, 2, 1.98f, 0.284f, 0.457f, 4.25f, 5.79f, 1.0f}, {32, 128, 256, 2, 2.14f, 0.357f, 0.560f, 4.88f, 5.78f, 1.0f},
};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);

TiledPlan tiled_plan(int m, int n, int k, int max_splits, bool swiglu, double* us_of_plan) {
    const int steps = (k + kTiledStep - 1) / kTiledStep, units = resident_waves() / 32;
    const double mn = (double)m * n, weight_bytes = 2.0 * n * k;
    TiledPlan best = {0, 1, steps};
    double best_us = 0.0;
    for (int c = 0; c < kTileCount; c++) {
        const TiledTile& tile = kTiles[c];
        // rows of a tile that do not exist are work for nothing; tiles of 32 rows read the weights once for each
        if ((tile.rows >= 2 * m && tile.rows > 32) || (tile.rows == 32 && m > 64)) continue;
        const int tiles = ((m + tile.rows - 1) / tile.rows) * ((n + tile.cols - 1) / tile.cols), slots = units * tile.per_unit;
        const double stream = 2.0 + weight_bytes / tile.stream_tb * 1e-6;
        for (int s = 1; s <= max_splits && (s == 1 || (2 * s <= steps && tiles * (s - 1) < slots)); s++) {  // more only fill a chip twice over
            const int per = (steps + s - 1) / s;
            if (s > 1 && per * (s - 1) >= steps) continue;  // the same as a smaller number
            const int groups = tiles * s, whole = groups / slots, rest = groups - whole * slots;
            const double longer = swiglu && s == 1 ? per * tile.swiglu : per;
            const double alone = tile.start_us + longer * tile.step_us, paired = tile.start_us + longer * tile.pair_us;
            double us;
            if (tile.per_unit == 1) us = (whole + (rest > 0)) * alone;
            else us = whole * paired + (rest > units ? paired : rest > 0 ? alone : 0.0);
            // partial sums: written here, and read (4.5 TB/s) in place of one fp16 value by whatever adds them up
            const double sums = s == 1 ? 0.0 : 4.0 * s * mn / tile.partial_tb * 1e-6 + (4.0 * s - 2.0) * mn / 4.5 * 1e-6;
            if (best_us > 0.0 && (us > stream ? us : stream) + sums >= best_us) continue;
            us = sqrt(sqrt(us * us * us * us + stream * stream * stream * stream)) + sums;
            if (best_us == 0.0 || us < best_us) {
                best_us = us;
                best = {c, s, per};
            }
        }
    }
    *us_of_plan = best_us;
    return best;
}

void tiled_extents(const TiledPlan& plan, int* rows, int* cols) {
    *rows = kTiles[plan.tile].rows;
    *cols = kTiles[plan.tile].cols;
}

template <int RESULT>
static void launch(const TiledPlan& plan, const __half* a, const __half* w, __half* out, float* partial, int m, int n, int k,
                   hipStream_t stream) {
    const TiledTile& tile = kTiles[plan.tile];
    const int cols = RESULT == kTiledSwiglu ? tile.cols / 2 : tile.cols, width = RESULT == kTiledSwiglu ? n / 2 : n;
    const dim3 grid((unsigned)((m + tile.rows - 1) / tile.rows) * (unsigned)((width + cols - 1) / cols), (unsigned)plan.splits);
#define ISP_TILED(INDEX, BM, BN, WM, WN, STAGES)                                                                              \
    case INDEX:                                                                                                               \
        static_assert(kTiles[INDEX].rows == BM && kTiles[INDEX].cols == BN && kTiles[INDEX].threads == kWave * WM * WN, "tile"); \
        hipLaunchKernelGGL((linear_tiled_f16<BM, BN, WM, WN, STAGES, RESULT>), grid, dim3(kWave * WM * WN), 0, stream, a, w,   \
                           out, partial, m, n, k, plan.steps_per_split);                                                      \
        break
    switch (plan.tile) {
        ISP_TILED(0, 256, 256, 2, 4, 2);
        ISP_TILED(1, 192, 256, 2, 4, 2);
        ISP_TILED(2, 256, 128, 4, 2, 3);
        ISP_TILED(3, 128, 256, 2, 4, 3);
        ISP_TILED(4, 128, 192, 2, 2, 2);
        ISP_TILED(5, 128, 128, 4, 2, 4);
        ISP_TILED(6, 128, 64, 2, 2, 3);
        ISP_TILED(7, 64, 128, 2, 2, 3);
        ISP_TILED(8, 64, 64, 2, 2, 4);
        ISP_TILED(9, 32, 128, 1, 4, 4);
    }
#undef ISP_TILED
}

void launch_tiled(const TiledPlan& plan, const __half* a, const __half* w, __half* out, float* partial, int m, int n, int k,
                  hipStream_t stream) {
    if (plan.splits > 1) launch<kTiledPartial>(plan, a, w, nullptr, partial, m, n, k, stream);
    else launch<kTiledHalf>(plan, a, w, out, nullptr, m, n, k, stream);
}

void launch_tiled_swiglu(const TiledPlan& plan, const __half* a, const __half* gate_up, __half* out, int m, int inter, int k,
                         hipStream_t stream) {
    launch<kTiledSwiglu>(plan, a, gate_up, out, nullptr, m, 2 * inter, k, stream);
}

}  // namespace isp
