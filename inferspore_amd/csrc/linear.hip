// isp_linear_rows_f16: the product of activation rows with a weight matrix, up to 16 rows by the kernel in linear_rows.h, more than 64 by the
// tiles in linear_tiled.h, between them by whichever is priced lower (product_plan); isp_linear_f16: up to 64 of them.
// The reference calls cuBLAS for it (src/kernels/linear.cu:7-66); the library here, hipBLASLt, reads the weights of a
// 16-row product at 1.4-3.8 TB/s and those of a 64-row product at 1.2-1.8 (4.9 for the widest), these kernels at 4.3-5.5
// and 3.1-5.4.
#include "linear_rows.h"

namespace isp {

void launch_skinny(const SkinnyPlan& plan, const __half* a, const __half* w, __half* out, float* partial, int m, int n, int k,
                   hipStream_t stream) {
    const dim3 grid((unsigned)plan.strips, (unsigned)plan.splits);
#define ISP_SKINNY(MT)                                                                                                    \
    if (out)                                                                                                              \
        hipLaunchKernelGGL((linear_skinny_f16<MT, false>), grid, dim3(kBlock), 0, stream, a, w, out, partial, m, n, k,    \
                           plan.steps_per_split);                                                                         \
    else                                                                                                                  \
        hipLaunchKernelGGL((linear_skinny_f16<MT, true>), grid, dim3(kBlock), 0, stream, a, w, out, partial, m, n, k,     \
                           plan.steps_per_split)
    if (m <= 16) ISP_SKINNY(1);
    else if (m <= 32) ISP_SKINNY(2);
    else if (m <= 48) ISP_SKINNY(3);
    else ISP_SKINNY(4);
#undef ISP_SKINNY
}

// out = fp16(sum over the splits, in their order); four columns per lane.
__global__ __launch_bounds__(kBlock) void linear_add_splits(const float* __restrict__ partial, __half* __restrict__ out,
                                                            unsigned quads, int splits) {
    const unsigned i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= quads) return;
    const float* const at[1] = {partial + 4 * (size_t)i};
    float4v sums[1];
    add_splits(at, 4 * (size_t)quads, splits, sums);
    const float4v sum = sums[0];
    const __half2 lo = __floats2half2_rn(sum[0], sum[1]), hi = __floats2half2_rn(sum[2], sum[3]);
    reinterpret_cast<uint2*>(out)[i] = make_uint2(*reinterpret_cast<const uint32_t*>(&lo), *reinterpret_cast<const uint32_t*>(&hi));
}

void launch_add_splits(const float* partial, int splits, __half* out, int m, int n, hipStream_t stream) {
    const unsigned quads = (unsigned)((size_t)m * (size_t)n / 4);
    hipLaunchKernelGGL(linear_add_splits, dim3((quads + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, partial, out, quads, splits);
}

// Extents that the kernels can count: a few rows, or any number of them (the addition below indexes four values in 32 bits).
static bool linear_shape(int m, int n, int k) {
    const int most = m <= kSkinnyMaxRows ? kSkinnyMaxExtent : kTiledMaxExtent;
    return k > 0 && n % 8 == 0 && k % 8 == 0 && n <= most && k <= most && m <= kTiledMaxRows && (long long)m * n < kTiledMaxValues;
}

static int linear(const __half* a, const __half* w, __half* out, float* workspace, int m, int n, int k, hipStream_t stream) {
    if (m < 0 || n < 0 || k < 0) return ISP_ERR_BAD_SHAPE;
    if (m == 0 || n == 0) return ISP_OK;
    if (!linear_shape(m, n, k)) return ISP_ERR_UNSUPPORTED;
    ISP_REQUIRE_PTR(a);
    ISP_REQUIRE_PTR(w);
    ISP_REQUIRE_PTR(out);
    if (!aligned16(a) || !aligned16(w) || !aligned16(out)) return ISP_ERR_UNSUPPORTED;
    const ProductPlan plan = product_plan(m, n, k);
    if (plan.splits() > 1) {
        ISP_REQUIRE_PTR(workspace);
        if (!aligned16(workspace)) return ISP_ERR_UNSUPPORTED;
    }
    launch_product(plan, a, w, out, workspace, m, n, k, stream);
    const int status = note_launch(hipGetLastError());
    if (status != ISP_OK || plan.splits() == 1) return status;
    launch_add_splits(workspace, plan.splits(), out, m, n, stream);
    return note_launch(hipGetLastError());
}

static int tell_plan(const ProductPlan& plan, int* tile_rows, int* tile_cols, int* splits) {
    ISP_REQUIRE_PTR(tile_rows);
    ISP_REQUIRE_PTR(tile_cols);
    ISP_REQUIRE_PTR(splits);
    *tile_rows = *tile_cols = 0;
    if (plan.tiled) tiled_extents(plan.tile, tile_rows, tile_cols);
    *splits = plan.splits();
    return ISP_OK;
}

}  // namespace isp

extern "C" {

size_t isp_linear_rows_f16_workspace(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || !isp::linear_shape(m, n, k)) return 0;
    const isp::ProductPlan plan = isp::product_plan(m, n, k);
    return plan.splits() == 1 ? 0 : plan.bytes(m, n);
}

int isp_linear_rows_f16(const void* a, const void* w, void* out, void* workspace, int m, int n, int k, isp_stream_t stream) {
    return isp::linear(static_cast<const __half*>(a), static_cast<const __half*>(w), static_cast<__half*>(out),
                       static_cast<float*>(workspace), m, n, k, static_cast<hipStream_t>(stream));
}

int isp_linear_rows_f16_plan(int m, int n, int k, int* tile_rows, int* tile_cols, int* splits) {
    if (m <= 0 || n <= 0 || k <= 0 || !isp::linear_shape(m, n, k)) return ISP_ERR_BAD_SHAPE;
    return isp::tell_plan(isp::product_plan(m, n, k), tile_rows, tile_cols, splits);
}

int isp_gate_up_rows_f16_plan(int m, int inter, int k, int* tile_rows, int* tile_cols, int* splits) {
    if (m <= 0 || inter <= 0 || k <= 0 || inter > isp::kTiledMaxExtent / 2 || inter % 8 != 0 || !isp::linear_shape(m, 2 * inter, k))
        return ISP_ERR_BAD_SHAPE;
    return isp::tell_plan(isp::product_plan(m, 2 * inter, k, isp::kTiledMaxSplits, true), tile_rows, tile_cols, splits);
}

size_t isp_linear_f16_workspace(int m, int n, int k) {
    if (m > isp::kSkinnyMaxRows) return 0;
    return isp_linear_rows_f16_workspace(m, n, k);
}

int isp_linear_f16(const void* a, const void* w, void* out, void* workspace, int m, int n, int k, isp_stream_t stream) {
    if (m > isp::kSkinnyMaxRows && n > 0 && k >= 0) return ISP_ERR_UNSUPPORTED;
    return isp_linear_rows_f16(a, w, out, workspace, m, n, k, stream);
}

}  // extern "C"
