// Fused causal attention for fp32 heads of 64, 96 or 128 elements, and for fp16 heads of 96 with few queries (the decode kernel of
// context_attention.hip wants powers of two), which are converted when they are loaded: what that file does for fp16, in fp32 throughout
// (v_mfma_f32_16x16x4_f32 multiplies and adds fp32; probabilities and sums stay fp32).  In place of KV broadcast, a mask tensor,
// torch's attention, two layout copies and the transpose to packed rows.
//
// A workgroup owns 16 queries: 16 neighbouring tokens of one head, or, where all heads of a group have at most 16
// queries together (a decode step), all of those, so that the group's keys are read once.  Its four wavefronts take every fourth
// block of 16 keys, straight from memory to registers, and are combined through LDS.  With j = lane % 16, g = lane / 16:
//   S^T[key, query] = K x Q^T   a product takes four d; which ones does not matter as long as both operands agree, so lane (j, g)
//                               loads the contiguous quarter d = HS / 4 g ... of key j and product i takes its element i;
//   O^T[d, query] = V^T x P^T   lane (j, g) holds the scores of query j and keys 4 g + r: product r takes keys 4 g + r, whose
//                               probabilities are the operand as they are; of value row 4 g + r the lane loads d = HS / 16 j ...
// Bound by the fp32 matrix rate (157 TFLOP/s) for long prompts and by the chain of dependent blocks for short ones.
// Against those five launches, us: 4 prompts of 100 tokens, 16 heads of 128: 11.0, 46.7; 1000 and 700 tokens, 32 heads over 8 key
// heads: 225, 887; 8 x 300 tokens on a history of 700, 32 heads: 650, 860; decode, 16 sequences of 1000 keys, 32 heads: 117, 449;
// 64 of 400, 32 heads of 96 over 8: 34, 343.  fp16 heads of 96: decode, 16 x 1000 keys, 32 heads 47, 140; 64 x 400, 32 over 8
// 26, 234; prompts beyond one workgroup per compute unit are the tiled kernel's.  Error against 64 bits 1.5e-7 ... 3.7e-7 (2-norm),
// there 2.1e-7 ... 6.9e-7.
#include <type_traits>

#include "isp_common.h"

namespace isp {

namespace {

typedef float float4w __attribute__((ext_vector_type(4)));

constexpr int kSlots = 16, kBlockKeys = 16, kWaves = 4;

__device__ __forceinline__ float rows_max(float x) {  // over the lanes of equal lane % 16
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// N elements from a 16-byte aligned address / two at a time, as fp32
template <int N>
__device__ __forceinline__ void load_row(const float* p, float* f) {
#pragma unroll
    for (int i = 0; i < N; i += 4) Elem<float>::unpack(load16(p + i), f + i);
}
template <int N>
__device__ __forceinline__ void load_row(const __half* p, float* f) {
#pragma unroll
    for (int i = 0; i < N; i += 8) Elem<__half>::unpack(load16(p + i), f + i);
}
template <int N>
__device__ __forceinline__ void load_pairs(const float* p, float* f) {
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        const float2 x = *reinterpret_cast<const float2*>(p + i);
        f[i] = x.x, f[i + 1] = x.y;
    }
}
template <int N>
__device__ __forceinline__ void load_pairs(const __half* p, float* f) {
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        const float2 x = __half22float2(*reinterpret_cast<const __half2*>(p + i));
        f[i] = x.x, f[i + 1] = x.y;
    }
}
__device__ __forceinline__ void store4(float* p, float4w x) { *reinterpret_cast<float4w*>(p) = x; }
__device__ __forceinline__ void store4(__half* p, float4w x) {
    reinterpret_cast<__half2*>(p)[0] = __floats2half2_rn(x[0], x[1]);
    reinterpret_cast<__half2*>(p)[1] = __floats2half2_rn(x[2], x[3]);
}

// GROUPED: the 16 queries are those of a group's heads (grid x = key head), else of 16 tokens of a head (x = head); grid y =
// sequence, z = tile of queries, the last (longest) first.
template <typename T, int HS, bool GROUPED>
__global__ __launch_bounds__(256) void context_attention_f32(
    const T* __restrict__ q_buf, const T* __restrict__ k_cache, const T* __restrict__ v_cache, T* __restrict__ out,
    const int* history_length, const int* input_length, const int* context_length, int head_num,
    int kv_head_num, int max_q_len, int max_k_len, int max_seq_len, int tokens, float scale_log2e) {
    constexpr int kQuarter = HS / 4, kChunk = HS / 16;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), j = lane % 16, g = lane / 16;
    const int b = blockIdx.y, group = head_num / kv_head_num;
    const int kv_head = GROUPED ? (int)blockIdx.x : (int)blockIdx.x / group;
    const int q0 = GROUPED ? 0 : (int)(gridDim.z - 1 - blockIdx.z) * kSlots;
    const int len = min(read_only_i32(input_length, b), max_q_len);
    if (q0 >= len) return;  // workgroup-uniform: padded queries only
    const int used = GROUPED ? group * len : min(kSlots, len - q0);  // slots with a query
    const int hist = read_only_i32(history_length, b);
    const int ctx = min(min(read_only_i32(context_length, b), max_k_len), max_seq_len);
    const int last_q = GROUPED ? len - 1 : q0 + used - 1;
    const int wg_visible = max(0, min(hist + last_q + 1, ctx));
    const bool real = j < used;
    const int my_q = !real ? q0 : GROUPED ? j / group : q0 + j;
    const int my_head = GROUPED ? kv_head * group + (real ? j % group : 0) : (int)blockIdx.x;
    const int my_visible = real ? min(hist + my_q + 1, ctx) : 0;
    const size_t kv_offset = ((size_t)b * kv_head_num + kv_head) * (size_t)max_seq_len * HS;
    const T *keys = k_cache + kv_offset, *values = v_cache + kv_offset;

    const int blocks = (wg_visible + kBlockKeys - 1) / kBlockKeys;
    float qf[kQuarter];
    if (wave < blocks) {  // a wavefront without keys has no use for the queries
        const T* q_row = q_buf + (((size_t)b * head_num + my_head) * (size_t)max_q_len + my_q) * HS + kQuarter * g;
        load_row<kQuarter>(q_row, qf);
#pragma unroll
        for (int i = 0; i < kQuarter; i++) qf[i] = real ? qf[i] : 0.0f;
    }
    float4w acc[kChunk];
#pragma unroll
    for (int c = 0; c < kChunk; c++) acc[c] = float4w{0.0f, 0.0f, 0.0f, 0.0f};
    float run_max = -INFINITY, run_sum = 0.0f;  // run_sum: this lane's keys only

    const auto block = [&](int s, auto tail) {
        // a key past the visible ones (in the last block only) re-reads the last visible row: its score is masked, its value counts as zero
        float kf[kQuarter], vf[4][kChunk];
        const T* k_row = keys + (size_t)min(s * kBlockKeys + j, wg_visible - 1) * HS + kQuarter * g;
        load_row<kQuarter>(k_row, kf);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const T* v_row = values + (size_t)min(s * kBlockKeys + 4 * g + r, wg_visible - 1) * HS + kChunk * j;
            load_pairs<kChunk>(v_row, vf[r]);
        }
        // two chains of products, so that one does not wait for the other's result
        float4w even = {0.0f, 0.0f, 0.0f, 0.0f}, odd = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < kQuarter; i += 2) {
            even = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], qf[i], even, 0, 0, 0);
            odd = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i + 1], qf[i + 1], odd, 0, 0, 0);
        }
        float p[4], m = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            p[r] = s * kBlockKeys + 4 * g + r < my_visible ? (even[r] + odd[r]) * scale_log2e : -INFINITY;
            m = fmaxf(m, p[r]);
        }
        const float new_max = fmaxf(run_max, rows_max(m));
        const float safe_max = new_max == -INFINITY ? 0.0f : new_max;  // no visible key yet
        // 1 also for a column without a query: its sum and accumulators are zero
        const float rescale = new_max == run_max ? 1.0f : __builtin_amdgcn_exp2f(run_max - safe_max);
        run_max = new_max;
        run_sum *= rescale;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            p[r] = __builtin_amdgcn_exp2f(p[r] - safe_max);
            run_sum += p[r];
        }
        if (__any(rescale != 1.0f)) {
#pragma unroll
            for (int c = 0; c < kChunk; c++) acc[c] *= rescale;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool exists = !decltype(tail)::value || s * kBlockKeys + 4 * g + r < wg_visible;  // 0 x inf is NaN
#pragma unroll
            for (int c = 0; c < kChunk; c++)
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(exists ? vf[r][c] : 0.0f, p[r], acc[c], 0, 0, 0);
        }
    };
    // every wavefront's last block is treated as a tail: contexts of a few blocks then run one copy of the code only
    int s = wave;
    for (; s + kWaves < blocks; s += kWaves) block(s, std::false_type{});
    if (s < blocks) block(s, std::true_type{});

    // O^T row 4 g + r of product c is d = kChunk (4 g + r) + c
    __shared__ __align__(16) float o_lds[kWaves][kSlots][HS];
    __shared__ float m_lds[kWaves][kSlots], l_lds[kWaves][kSlots];
    run_sum = rows_sum(run_sum);
    if (g == 0) {
        m_lds[wave][j] = run_max;
        l_lds[wave][j] = run_sum;
    }
    if (real) {
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int c = 0; c < kChunk; c += 2)
                *reinterpret_cast<float2*>(&o_lds[wave][j][kChunk * (4 * g + r) + c]) = make_float2(acc[c][r], acc[c + 1][r]);
    }
    __shared__ int length_shares[kWaves];
    sum_lengths_wave(sum_lengths_thread(input_length, b), b, length_shares);
    __syncthreads();
    const int first_token = sum_lengths_total(length_shares);
    for (int at = tid; at < used * (HS / 4); at += 256) {
        const int slot = at / (HS / 4), d = 4 * (at % (HS / 4));
        float m = m_lds[0][slot];
#pragma unroll
        for (int w = 1; w < kWaves; w++) m = fmaxf(m, m_lds[w][slot]);
        const float safe = m == -INFINITY ? 0.0f : m;
        float4w o = {0.0f, 0.0f, 0.0f, 0.0f};
        float l = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const float e = __builtin_amdgcn_exp2f(m_lds[w][slot] - safe);
            l += e * l_lds[w][slot];
            o += e * *reinterpret_cast<const float4w*>(&o_lds[w][slot][d]);
        }
        const int head = GROUPED ? kv_head * group + slot % group : (int)blockIdx.x;
        const long long token = (long long)first_token + (GROUPED ? slot / group : q0 + slot);
        if (token < tokens)
            store4(out + ((size_t)token * head_num + head) * HS + d, o * (l > 0.0f ? 1.0f / l : 0.0f));
    }
}

}  // namespace

template <typename T>
static int attention_f32(const T* q, const T* k_cache, const T* v_cache, T* out, const int32_t* history_length,
                         const int32_t* input_length, const int32_t* context_length, int layer, int batch, int head_num,
                         int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int token_num, float scale,
                         hipStream_t stream) {
    if (layer < 0 || batch < 0 || head_num <= 0 || kv_head_num <= 0 || head_num % kv_head_num != 0 || max_q_len < 0 ||
        max_k_len < 0 || max_seq_len < 0 || token_num < 0 || !(scale > 0.0f))
        return ISP_ERR_BAD_SHAPE;
    if (head_size != 96 && (sizeof(T) == 2 || (head_size != 128 && head_size != 64))) return ISP_ERR_UNSUPPORTED;
    if (batch == 0 || max_q_len == 0 || token_num == 0) return ISP_OK;
    if (max_k_len == 0 || max_seq_len == 0) return ISP_ERR_BAD_SHAPE;
    const bool grouped = (long long)(head_num / kv_head_num) * max_q_len <= kSlots;
    const int tiles = grouped ? 1 : (max_q_len + kSlots - 1) / kSlots;
    if (batch > 65535 || tiles > 65535) return ISP_ERR_UNSUPPORTED;
    ISP_REQUIRE_PTR(q);
    ISP_REQUIRE_PTR(k_cache);
    ISP_REQUIRE_PTR(v_cache);
    ISP_REQUIRE_PTR(out);
    ISP_REQUIRE_PTR(history_length);
    ISP_REQUIRE_PTR(input_length);
    ISP_REQUIRE_PTR(context_length);
    if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out)) return ISP_ERR_UNSUPPORTED;
    const size_t slice = (size_t)layer * batch * kv_head_num * max_seq_len * head_size;
    const dim3 grid((unsigned)(grouped ? kv_head_num : head_num), (unsigned)batch, (unsigned)tiles);
#define ISP_LAUNCH_F32(HS, GROUPED)                                                                                          \
    hipLaunchKernelGGL((context_attention_f32<T, HS, GROUPED>), grid, dim3(256), 0, stream, q, k_cache + slice, v_cache + slice, out, \
                       history_length, input_length, context_length, head_num, kv_head_num, max_q_len, max_k_len,            \
                       max_seq_len, token_num, scale * 1.4426950408889634f)
#define ISP_LAUNCH_F32_HS(HS)               \
    do {                                    \
        if (grouped) ISP_LAUNCH_F32(HS, true); \
        else ISP_LAUNCH_F32(HS, false);     \
    } while (0)
    if constexpr (sizeof(T) == 2) {
        ISP_LAUNCH_F32_HS(96);
    } else {
        if (head_size == 128) ISP_LAUNCH_F32_HS(128);
        else if (head_size == 96) ISP_LAUNCH_F32_HS(96);
        else ISP_LAUNCH_F32_HS(64);
    }
#undef ISP_LAUNCH_F32_HS
#undef ISP_LAUNCH_F32
    return note_launch(hipGetLastError());
}

int context_attention_f16_96(const __half* q, const __half* k_cache, const __half* v_cache, __half* out,
                             const int32_t* history_length, const int32_t* input_length, const int32_t* context_length, int layer,
                             int batch, int head_num, int kv_head_num, int max_q_len, int max_k_len, int max_seq_len,
                             int token_num, float scale, hipStream_t stream) {
    return attention_f32<__half>(q, k_cache, v_cache, out, history_length, input_length, context_length, layer, batch, head_num,
                                 kv_head_num, 96, max_q_len, max_k_len, max_seq_len, token_num, scale, stream);
}

}  // namespace isp

extern "C" int isp_context_attention_f32(const void* q, const void* k_cache, const void* v_cache, void* out,
                                         const int32_t* history_length, const int32_t* input_length,
                                         const int32_t* context_length, int layer, int batch, int head_num,
                                         int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len,
                                         int token_num, float scale, isp_stream_t stream) {
    return isp::attention_f32<float>(static_cast<const float*>(q), static_cast<const float*>(k_cache),
                              static_cast<const float*>(v_cache), static_cast<float*>(out), history_length, input_length,
                              context_length, layer, batch, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                              max_seq_len, token_num, scale, static_cast<hipStream_t>(stream));
}
