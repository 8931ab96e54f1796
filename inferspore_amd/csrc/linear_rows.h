// Skinny product of a layer: C[m, n] = A[m, k] x W[k, n], fp16, row-major, fp32 accumulation, for the few rows of a
// decode step or a short prompt.  The weights are read once and bound the time; everything below serves that one stream.
//
// A wavefront owns 128 columns and takes 32 rows of W per step: lane (j = lane % 16, g = lane / 16) loads the eight
// columns 8 j ... 8 j + 7 of the eight rows 8 g ... 8 g + 7, so that every load instruction covers four whole 256-byte row
// segments and nothing goes through LDS.  Matrix cores want, per lane, eight consecutive k of ONE column
// (v_mfma_f32_16x16x32_f16): an 8 x 8 transpose inside the lane's own registers, one byte-permute per result dword.  Product c
// (0 ... 7) then takes column 8 j + c of every lane, and a lane ends with eight neighbouring columns of its output rows.
// The wavefronts of a workgroup take every WAVES-th step of the workgroup's k range and add up through LDS in a fixed
// order; workgroups that share a strip of columns write fp32 partial sums [splits][m][n] that the consumer adds in order.
#pragma once

#include <math.h>

#include "isp_common.h"

namespace isp {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kStripCols = 128;  // columns of a workgroup
constexpr int kStepRows = 32;    // rows of W per step of a wavefront

struct SkinnyStep {
    vec16 w[8];
};

// Column c of the lane's 8 x 8 block as one operand: dword i holds rows 2 i and 2 i + 1.
__device__ __forceinline__ half8 block_column(const SkinnyStep& t, int c) {
    union { uint32_t u[4]; half8 h; } r;
#pragma unroll
    for (int i = 0; i < 4; i++)
        r.u[i] = __builtin_amdgcn_perm(t.w[2 * i + 1].w[c / 2], t.w[2 * i].w[c / 2], c % 2 ? 0x07060302u : 0x05040100u);
    return r.h;
}

// MT: tiles of 16 rows of A.  SPLIT: fp32 partial sums to `partial`, else fp16 to `out`.
template <int MT, bool SPLIT>
__global__ __launch_bounds__(kBlock) void linear_skinny_f16(const __half* __restrict__ a, const __half* __restrict__ w,
                                                                 __half* __restrict__ out, float* __restrict__ partial, int m,
                                                                 int n, int k, int steps_per_split) {
    constexpr int WAVES = kBlock / kWave;
    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane % 16, g = lane / 16;
    const int strip0 = (int)blockIdx.x * kStripCols;
    const int steps = (k + kStepRows - 1) / kStepRows;
    const int first = (int)blockIdx.y * steps_per_split, last = min(steps, first + steps_per_split);
    // lanes past the last column (row of A past m) read the last ones that exist; their results are not stored
    const __half* w_lane = w + min(strip0 + 8 * j, n - 8);
    const __half* a_lane[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) a_lane[t] = a + (size_t)min(16 * t + j, m - 1) * (size_t)k;

    float4v acc[MT][8];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int c = 0; c < 8; c++) acc[t][c] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    SkinnyStep buf[2];
    half8 af[2][MT];
    auto load = [&](int which, int s) {
        // k is a multiple of 8, so a lane's eight rows exist together or not at all (last step only)
        const int row = min(s * kStepRows + 8 * g, k - 8);
        const __half* p = w_lane + (size_t)row * (size_t)n;
#pragma unroll
        for (int i = 0; i < 8; i++) buf[which].w[i] = load16_stream(p + (size_t)i * (size_t)n);
#pragma unroll
        for (int t = 0; t < MT; t++) af[which][t] = *reinterpret_cast<const half8*>(a_lane[t] + row);
    };
    auto compute = [&](int which, int s) {
        if ((s + 1) * kStepRows > k) {  // wavefront-uniform: rows past k count as zero on both sides (0 x inf is NaN)
            const uint32_t keep = s * kStepRows + 8 * g < k ? 0xffffffffu : 0u;
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) buf[which].w[i].w[e] &= keep;
#pragma unroll
            for (int t = 0; t < MT; t++)
                if (!keep) af[which][t] = half8{0, 0, 0, 0, 0, 0, 0, 0};
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const half8 b = block_column(buf[which], c);
#pragma unroll
            for (int t = 0; t < MT; t++) acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[which][t], b, acc[t][c], 0, 0, 0);
        }
    };
    // The next step's loads are in flight while a step is computed.  No load sits behind a branch that joins again (how many
    // are outstanding would no longer be known, and every one would be waited for): each half of the loop has its own way
    // out.  A third or fourth step in flight measured the same at 16 rows and spills registers from 48 rows on.
    int s = first + wave;
    if (s < last) {
        load(0, s);
        for (;;) {
            if (s + WAVES >= last) {
                compute(0, s);
                break;
            }
            load(1, s + WAVES);
            compute(0, s);
            s += WAVES;
            if (s + WAVES >= last) {
                compute(1, s);
                break;
            }
            load(0, s + WAVES);
            compute(1, s);
            s += WAVES;
        }
    }

    // 16 rows at a time through LDS: lane (j, g) holds rows 4 g + r and columns 8 j + c
    __shared__ __align__(16) float tile[WAVES][16][kStripCols];
    constexpr int elems = 16 * kStripCols / kBlock;  // floats a thread adds up: 8
    const int row = tid * elems / kStripCols, col = tid * elems % kStripCols;
#pragma unroll
    for (int t = 0; t < MT; t++) {
        if (t > 0) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                *reinterpret_cast<float4v*>(&tile[wave][4 * g + r][8 * j + 4 * h]) =
                    float4v{acc[t][4 * h][r], acc[t][4 * h + 1][r], acc[t][4 * h + 2][r], acc[t][4 * h + 3][r]};
        __syncthreads();
        const int out_row = 16 * t + row, out_col = strip0 + col;
        if (out_row < m && out_col < n) {  // n is a multiple of 8: a thread's columns exist together
#pragma unroll
            for (int e = 0; e < elems; e += 4) {
                float4v sum = *reinterpret_cast<const float4v*>(&tile[0][row][col + e]);
#pragma unroll
                for (int v = 1; v < WAVES; v++) sum += *reinterpret_cast<const float4v*>(&tile[v][row][col + e]);
                const size_t at = (size_t)out_row * (size_t)n + (size_t)(out_col + e);
                if (SPLIT) {
                    *reinterpret_cast<float4v*>(partial + (size_t)blockIdx.y * (size_t)m * (size_t)n + at) = sum;
                } else {
                    const __half2 lo = __floats2half2_rn(sum[0], sum[1]), hi = __floats2half2_rn(sum[2], sum[3]);
                    *reinterpret_cast<uint2*>(out + at) = make_uint2(*reinterpret_cast<const uint32_t*>(&lo), *reinterpret_cast<const uint32_t*>(&hi));
                }
            }
        }
    }
}

// How many workgroups share a strip of columns.  Two costs are weighed: the rounds of one workgroup per compute unit that
// strips x splits make, over those that whole rounds would make (idle units at the end), and the partial sums, whose bytes
// are 2 m splits / k of the weights', written once and read back once.  The factor 4 in front of that ratio (2 would be the
// bytes alone) is what the measured plans want: the reading kernel depends on the last of them.  Measured with 16
// rows: 96 strips of 4096 rows (100.7 MB) 1, 2, 3, 4, 5, 8 splits 30.0, 19.4, 24.7, 20.5, 18.5, 19.0 us (taken: 5); 32
// strips (33.6 MB) 4, 8, 16 splits 9.9, 7.8, 7.7 (8); 172 strips 1, 2, 4 splits 34.7, 37.9, 32.5 (4).  With 64 rows: 32
// strips 4, 8, 16 splits 14.7, 11.3, 15.9 (8); 224 strips 1, 2 splits 49.7, 57.2 (1).  Every wavefront keeps a step, except in a
// last split that rounding up the others' steps leaves short.
struct SkinnyPlan {
    int strips, splits, steps_per_split;
    size_t partial_floats(int m, int n) const { return (size_t)splits * (size_t)m * (size_t)n; }
};
constexpr int kSkinnyMaxRows = 64, kSkinnyMaxSplits = 16;
constexpr int kSkinnyMaxExtent = 1 << 24;  // of n and k: the kernel counts columns, rows and results in 32 bits
inline SkinnyPlan skinny_plan(int m, int n, int k) {
    SkinnyPlan p;
    const int steps = (k + kStepRows - 1) / kStepRows, waves = kBlock / kWave, units = resident_waves() / 32;
    p.strips = (n + kStripCols - 1) / kStripCols;
    p.steps_per_split = steps;
    double best = 0.0;
    for (int s = 1; s <= kSkinnyMaxSplits && (s == 1 || s * waves <= steps); s++) {
        const long long groups = (long long)p.strips * s, rounds = (groups + units - 1) / units;
        const double cost = (double)(rounds * units) / (double)groups + 8.0 * (double)m * (double)s / (double)k;
        if (s == 1 || cost < best) {
            best = cost;
            p.steps_per_split = (steps + s - 1) / s;
        }
    }
    p.splits = (steps + p.steps_per_split - 1) / p.steps_per_split;
    return p;
}

// Partial sums of the product to `partial`, or with `out` (one split only) the fp16 product itself.  Operands checked by the caller.
void launch_skinny(const SkinnyPlan& plan, const __half* a, const __half* w, __half* out, float* partial, int m, int n, int k,
                   hipStream_t stream);

// Products of more rows (linear_tiled.h): which of the tiles, and how many workgroups share a tile's k.
struct TiledPlan {
    int tile, splits, steps_per_split;
};
// `us`: what the plan is estimated to take, the reading of its splits by whatever adds them included.
TiledPlan tiled_plan(int m, int n, int k, int max_splits, bool swiglu, double* us);
void tiled_extents(const TiledPlan& plan, int* rows, int* cols);
constexpr int kTiledMaxSplits = 16;
constexpr int kTiledMaxExtent = 1 << 22;  // of n and k: a tile's rows of A and of W are addressed in 32 bits
// of m: the tiles of the fewest rows, 64 in fp16 and 32 in fp32, times 256 threads make a grid that can be launched
constexpr int kTiledMaxRows = (1 << 30) - 1, kTiledMaxRowsF32 = (1 << 29) - 1;
constexpr long long kTiledMaxValues = 0x3ffffff00ll;  // m n: the addition of splits counts four values in 32 bits
// With plan.splits > 1 partial sums to `partial`, else the fp16 product to `out`.  Operands checked by the caller.
void launch_tiled(const TiledPlan& plan, const __half* a, const __half* w, __half* out, float* partial, int m, int n, int k,
                  hipStream_t stream);
// out[m, inter] = SwiGLU of the product with gate_up [k, 2 inter]; a plan without splits
void launch_tiled_swiglu(const TiledPlan& plan, const __half* a, const __half* gate_up, __half* out, int m, int inter, int k,
                         hipStream_t stream);

// The same in fp32 (linear_tiled_f32.h).  `us`: what the plan is estimated to take, the addition of its splits included.
TiledPlan tiled_plan_f32(int m, int n, int k, int max_splits, double* us);
void launch_tiled_f32(const TiledPlan& plan, const float* a, const float* w, float* out_or_partial, int m, int n, int k, hipStream_t stream);
// out[m, inter] = SwiGLU of the product with gate_up [k, 2 inter]; a plan without splits
void launch_tiled_swiglu_f32(const TiledPlan& plan, const float* a, const float* gate_up, float* out, int m, int inter, int k,
                             hipStream_t stream);

// Either, for the rows that it is made for.  A skinny product's sums end in the order of its wavefronts, a tiled one's in the order of k.
struct ProductPlan {
    bool tiled;
    SkinnyPlan skinny;
    TiledPlan tile;
    int splits() const { return tiled ? tile.splits : skinny.splits; }
    // what the product leaves for its consumer: fp16, or the splits' partial sums
    size_t bytes(int m, int n) const {
        const size_t values = (size_t)m * (size_t)n;
        return splits() == 1 ? values * sizeof(__half) : (size_t)splits() * values * sizeof(float);
    }
};
constexpr int kSkinnyRows = 16;  // the skinny kernel up to here, up to kSkinnyMaxRows whichever is priced lower
// What a skinny product of 17 ... 64 rows takes, the reading of its splits included: rounds of one workgroup per compute unit, each start +
// step per 128 k, against the weights' stream.  Fitted (mean error 3 to 4 %) to 1008 products of 17 to 64 rows, 1024 to 32768 columns and
// 1024 to 14336 k.
inline double skinny_us(const SkinnyPlan& plan, int m, int n, int k) {
    constexpr double kStart[] = {4.3, 4.64, 4.93}, kStep[] = {0.648, 1.033, 1.209}, kStream[] = {6.47, 6.75, 6.82};
    const int t = m <= 32 ? 0 : m <= 48 ? 1 : 2, waves = kBlock / kWave, units = resident_waves() / 32;
    const double mn = (double)m * n, stream = 2.0 + 2.0 * n * k / kStream[t] * 1e-6;
    const long long rounds = ((long long)plan.strips * plan.splits + units - 1) / units;
    const double us = (double)rounds * (kStart[t] + (plan.steps_per_split + waves - 1) / waves * kStep[t]);
    const double sums = plan.splits == 1 ? 0.0 : 4.0 * plan.splits * mn / 5.5 * 1e-6 + (4.0 * plan.splits - 2.0) * mn / 4.5 * 1e-6;
    return sqrt(sqrt(us * us * us * us + stream * stream * stream * stream)) + sums;
}
// swiglu: a plan without splits computes SwiGLU
inline ProductPlan product_plan(int m, int n, int k, int max_splits = kTiledMaxSplits, bool swiglu = false) {
    ProductPlan p = {m > kSkinnyRows, {}, {}};
    if (m <= kSkinnyMaxRows) p.skinny = skinny_plan(m, n, k);
    if (!p.tiled) return p;
    double us;
    p.tile = tiled_plan(m, n, k, max_splits, swiglu, &us);
    if (m > kSkinnyMaxRows) return p;
    // The skinny kernel reads the weights straight to registers, 5.8 to 6.5 TB/s where its strips fill whole rounds of compute units; the tiled
    // one needs no whole rounds and feeds more rows.  us, skinny and tiled, additions included: 17 x 4096 x 28672 39.5, 43.1; 32 x 8192 x
    // 8192 27.6, 30.7; 17 x 8192 x 32768 87.0, 91.2; 48 x 4096 x 12288 26.4, 24.1; 32 x 4096 x 22016 43.3, 36.0; 64 x 4096 x 28672 49.5,
    // 43.3.  The tiles' prices are 1.11 to 1.18 times what they take here, and what the skinny kernel
    // saves with the third and fourth tile of rows is less sure, hence the factors.  SwiGLU inside a tiled product saves a launch (3 us), but
    // reads two narrower streams, slowest where rows are whole multiples of 2 KiB: 17 x 4096 x 28672 49.7 against 39.8 and 5.0; a whole
    // layer of 48 rows x 4096, inter 11008, 125 against 131.  261 layers of 512 to 8192 columns take 0.2 % more than with the better of both
    // for each; at worst 2.3 % more than all skinny (which are up to 24 % slower) and 1.7 % more than all tiled (up to 14 %).
    double tiled = (m <= 32 ? 0.9 : m <= 48 ? 0.86 : 0.76) * us, skinny = skinny_us(p.skinny, m, n, k);
    if (swiglu && p.tile.splits == 1) {
        tiled *= 2ll * n % 2048 == 0 ? 1.28 : 1.05;
        skinny += 3.0;
    }
    p.tiled = tiled < skinny;
    return p;
}
// With several splits their sums to `partial`, else the fp16 product to `out`.
inline void launch_product(const ProductPlan& plan, const __half* a, const __half* w, __half* out, float* partial, int m, int n, int k,
                           hipStream_t stream) {
    if (plan.tiled) launch_tiled(plan.tile, a, w, out, partial, m, n, k, stream);
    else launch_skinny(plan.skinny, a, w, plan.skinny.splits == 1 ? out : nullptr, partial, m, n, k, stream);
}

// Values of a product left as partial sums, four neighbouring ones at each of p[0 ... PIECES): the splits added in their order.  `stride`:
// floats between two splits.  All loads of up to eight splits are on their way before the first is added (those past the last re-read
// it): the sums were just written by other XCDs, and a loop that waits for one load after the other took most of its kernel's time.
template <int CHUNK, int PIECES>
__device__ __forceinline__ void add_split_chunks(const float* const (&p)[PIECES], size_t stride, int splits, float4v (&sum)[PIECES]) {
    for (int s0 = 0; s0 < splits; s0 += CHUNK) {
        float4v v[CHUNK][PIECES];
#pragma unroll
        for (int s = 0; s < CHUNK; s++)
#pragma unroll
            for (int i = 0; i < PIECES; i++) v[s][i] = *reinterpret_cast<const float4v*>(p[i] + (size_t)min(s0 + s, splits - 1) * stride);
#pragma unroll
        for (int s = 0; s < CHUNK; s++)
#pragma unroll
            for (int i = 0; i < PIECES; i++) asm volatile("" : "+v"(v[s][i]));  // or the compiler moves each load behind the test below
#pragma unroll
        for (int s = 0; s < CHUNK; s++) {
            if (s0 + s >= splits) break;  // uniform
#pragma unroll
            for (int i = 0; i < PIECES; i++) sum[i] = s0 + s == 0 ? v[s][i] : sum[i] + v[s][i];
        }
    }
}
template <int PIECES>
__device__ __forceinline__ void add_splits(const float* const (&p)[PIECES], size_t stride, int splits, float4v (&sum)[PIECES]) {
    if (splits <= 4) add_split_chunks<4>(p, stride, splits, sum);  // uniform
    else add_split_chunks<8>(p, stride, splits, sum);
}
// Eight neighbouring columns rounded to fp16 once, the value linear_add_splits would have stored.
__device__ __forceinline__ vec16 pack_sums(const float4v& a, const float4v& b) {
    const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return Elem<__half>::pack(f);
}
__device__ __forceinline__ vec16 add_splits8(const float* p, size_t stride, int splits) {
    const float* const at[2] = {p, p + 4};
    float4v sum[2];
    add_splits(at, stride, splits, sum);
    return pack_sums(sum[0], sum[1]);
}
// 16 bytes of the product that the splits make up
template <typename T>
__device__ __forceinline__ vec16 add_splits_vector(const float* p, size_t stride, int splits) {
    if constexpr (sizeof(T) == 2) {
        return add_splits8(p, stride, splits);
    } else {
        const float* const at[1] = {p};
        float4v sum[1];
        add_splits(at, stride, splits, sum);
        const float f[4] = {sum[0][0], sum[0][1], sum[0][2], sum[0][3]};
        return Elem<float>::pack(f);
    }
}
__device__ __forceinline__ void add_splits8(const float* p, const float* q, size_t stride, int splits, vec16& first, vec16& second) {
    const float* const at[4] = {p, p + 4, q, q + 4};
    float4v sum[4];
    add_splits(at, stride, splits, sum);
    first = pack_sums(sum[0], sum[1]);
    second = pack_sums(sum[2], sum[3]);
}

// out[m][n] = the splits' sum, rounded to fp16.  n is a multiple of 8, m n / 4 fits 32 bits.
void launch_add_splits(const float* partial, int splits, __half* out, int m, int n, hipStream_t stream);

// Consumers of partial sums: what the entry points of the same step do with a stored fp16 product (same bits), with that
// product's addition of splits, its store and its read back taken out.  Operands checked by the caller.
void launch_qkv_sums(const float* partial, int splits, const __half* bias, __half* q, __half* k_cache, __half* v_cache,
                     const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length, int batch,
                     int seq_len, int tokens, int head_num, int kv_head_num, int head_size, int max_seq_len, int rot, float base,
                     hipStream_t stream);
template <typename T>
void launch_norm_sums(const float* partial, int splits, T* residual, T* out, const T* gamma, float eps, int tokens, int hidden,
                      hipStream_t stream);
constexpr int kNormSumsMaxHidden = 8192;  // in fp16: a vector per lane
void launch_swiglu_sums(const float* partial, int splits, __half* out, int tokens, int inter, hipStream_t stream);

// csrc/context_attention.hip
size_t attention_workspace(int batch, int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len);
int context_attention(const _Float16* q, const _Float16* k_cache, const _Float16* v_cache, _Float16* out,
                      const int32_t* history_length, const int32_t* input_length, const int32_t* context_length,
                      int layer, int batch, int head_num, int kv_head_num, int head_size, int max_q_len,
                      int max_k_len, int max_seq_len, int token_num, float scale, float* workspace, hipStream_t stream);

}  // namespace isp
