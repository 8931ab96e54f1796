// RMSNorm and fused add-residual + RMSNorm for launches of a few rows -- every decode-step norm, and prefill
// batches up to the size whose waves are all resident at once -- on gfx950.
// Semantics and row algorithm: norm_rows.h (src/kernels/fused_addresidual_norm.cu:55-97 in the reference).
// This file is built with kernel-argument preloading like the other kernel files: the arguments arrive in scalar
// registers with the wave instead of being fetched by its first instructions, one round trip less in a launch
// that is nothing but a chain of round trips (64 x 4096 fp32: 2.40 against 2.64 us per launch; 256 rows 3.2
// against 3.4).  The general kernel (norm.hip) is built without it: the benchmark configuration, 2048 x 4096
// fp16 with residual and bias in one round of waves, measured 1 % slower with it.
#include "linear_rows.h"
#include "norm_rows.h"

namespace isp {

// The same row algorithm for launches of a few rows (every decode-step norm).  Such a launch is a chain of
// latencies, not a stream: the device is mostly empty, nothing hides an instruction, and what the general
// kernel pays for deciding at run time which operands exist and in which order to store (branches, selects,
// and waits that must assume the worst because loads sit inside branches) is on the critical path -- 64 x
// 4096 fp32: 2.9 us per launch back to back with the general kernel, 2.6 us with the operands fixed at
// compile time, 2.4 us with the arguments preloaded as well, against 2.0 us for a copy of the same bytes.  One row per workgroup of WPR waves, one or two
// vectors per lane, the default residual order only.  Same operations in the same order, so the same bits.
// (Requesting gamma and bias together with the row, to take a cache round trip out of the chain, measured
// 0.05-0.2 us SLOWER at 16-256 rows, twice, in this kernel and in a stripped-down one.)
template <typename T, int NV, int WPR, int ST, int OPS>
__global__ __launch_bounds__(norm_block(WPR)) void fused_norm_few_rows(T* residual, T* out, const T* bias,
                                                                       const T* gamma, float eps, int tokens,
                                                                       int hidden) {
    norm_rows_body<T, NV, WPR, ST, norm_block(WPR), OPS>(residual, out, bias, gamma, eps, tokens, hidden, 0u);
}

template <typename T, int NV, int WPR, int ST>
static NormFewKernel<T> few_ops(int ops) {
    if (ops == kOpsNone) return fused_norm_few_rows<T, NV, WPR, ST, kOpsNone>;
    if (ops == kOpsResidual) return fused_norm_few_rows<T, NV, WPR, ST, kOpsResidual>;
    return fused_norm_few_rows<T, NV, WPR, ST, kOpsResidualBias>;
}

template <typename T>
NormFewKernel<T> norm_few_variant(int wpr, int nv, int st, int ops) {
    if (st != kStorePlain && st != kStoreStream) return nullptr;
    const bool plain = st == kStorePlain;
    if (nv == 2 && wpr == 16)
        return plain ? few_ops<T, 2, 16, kStorePlain>(ops) : few_ops<T, 2, 16, kStoreStream>(ops);
    if (nv != 1) return nullptr;
    switch (wpr) {
        case 1: return plain ? few_ops<T, 1, 1, kStorePlain>(ops) : few_ops<T, 1, 1, kStoreStream>(ops);
        case 2: return plain ? few_ops<T, 1, 2, kStorePlain>(ops) : few_ops<T, 1, 2, kStoreStream>(ops);
        case 4: return plain ? few_ops<T, 1, 4, kStorePlain>(ops) : few_ops<T, 1, 4, kStoreStream>(ops);
        case 8: return plain ? few_ops<T, 1, 8, kStorePlain>(ops) : few_ops<T, 1, 8, kStoreStream>(ops);
        case 16: return plain ? few_ops<T, 1, 16, kStorePlain>(ops) : few_ops<T, 1, 16, kStoreStream>(ops);
        default: return nullptr;
    }
}

template NormFewKernel<float> norm_few_variant<float>(int, int, int, int);
template NormFewKernel<__half> norm_few_variant<__half>(int, int, int, int);

// Residual + RMSNorm of a product left as partial sums [splits][tokens][hidden]: a row per workgroup, one vector per lane;
// the operations and their order are norm_rows_body's (absent waves add exact zeros), so the bits are too.
template <typename T>
__global__ __launch_bounds__(1024) void fused_norm_sums(const float* __restrict__ partial, int splits, T* __restrict__ residual,
                                                        T* __restrict__ out, const T* __restrict__ gamma, float eps, int tokens,
                                                        int hidden) {
    constexpr int VEC = Elem<T>::kVec;
    __shared__ float sums[16];
    const int tid = threadIdx.x, waves = blockDim.x / kWave;
    const bool ok = tid * VEC < hidden;
    const size_t at = (size_t)blockIdx.x * (size_t)hidden + (size_t)(ok ? tid : 0) * (unsigned)VEC;
    const vec16 vr = load16(residual + at), vg = load16(gamma + (ok ? tid : 0) * VEC);
    const vec16 vo = add_splits_vector<T>(partial + at, (size_t)tokens * (size_t)hidden, splits);
    float x[VEC];
    Elem<T>::sum(vo, vr, x);
#pragma unroll
    for (int e = 0; e < VEC; e++) x[e] = Elem<T>::pinned(x[e]);
    float p = x[0] * x[0];
#pragma unroll
    for (int e = 1; e < VEC; e++) p = __fmaf_rn(x[e], x[e], p);
    p = wave_sum(ok ? p : 0.0f);
    if (tid % kWave == 0) sums[tid / kWave] = p;
    __syncthreads();
    float part[16];
#pragma unroll
    for (int w = 0; w < 16; w++) part[w] = w < waves ? sums[w] : 0.0f;
    const float inv = rsqrtf(tree_sum<16>(part) / (float)hidden + eps);
    if (!ok) return;
    store16(residual + at, Elem<T>::pack_pinned(x));
    float y[VEC];
    Elem<T>::scale(vg, x, y);
#pragma unroll
    for (int e = 0; e < VEC; e++) y[e] *= inv;
    store16(out + at, Elem<T>::pack(y));
}

template <typename T>
void launch_norm_sums(const float* partial, int splits, T* residual, T* out, const T* gamma, float eps, int tokens, int hidden,
                      hipStream_t stream) {
    const unsigned threads = (unsigned)((hidden / Elem<T>::kVec + kWave - 1) / kWave * kWave);
    hipLaunchKernelGGL(fused_norm_sums<T>, dim3((unsigned)tokens), dim3(threads), 0, stream, partial, splits, residual, out, gamma,
                       eps, tokens, hidden);
}
template void launch_norm_sums<__half>(const float*, int, __half*, __half*, const __half*, float, int, int, hipStream_t);
template void launch_norm_sums<float>(const float*, int, float*, float*, const float*, float, int, int, hipStream_t);

}  // namespace isp
