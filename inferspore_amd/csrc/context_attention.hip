// Fused causal attention of a context-decoder layer for fp16 heads of 128, 96 or 64 elements: one kernel in place of
// KV broadcast, q x k^T, masked softmax, p x v and the transpose back to packed tokens.  It reads the padded
// queries [batch, head_num, max_q_len, hs], the layer's slice of the KV cache [batch, kv_head_num,
// max_seq_len, hs] (keys and values of the history and of this call's tokens) and writes the packed
// [tokens, head_num, hs] rows the output projection consumes.  The [queries x keys] scores never leave the
// registers, and key tiles behind the causal diagonal are not visited.
//
// The mask is the one of the layer's softmax: query q of sequence b sees the keys at positions
// < min(history_length[b] + q + 1, context_length[b], max_k_len).  A deliberate departure from the reference when a
// sequence has history: its mask (src/kernels/build_casual_mask.cu:36) additionally requires k >= context length -
// query length, which hides every history key -- the comment above that line calls it the mask that does not support
// multi-turn dialogue and draws the one that does, which is the one computed here.  With history_length = 0 the two
// are the same mask.
//
// Matrix cores: v_mfma_f32_32x32x16_f16.  A wavefront owns 32 queries.  It computes the TRANSPOSED scores
// S^T[key, query] = K x Q^T, so that a lane's 16 accumulators of a 32 x 32 block all belong to one query
// (column = lane % 32): the running maximum and sum of the online softmax are per-lane scalars, combined only
// with the other half of the wavefront (lane ^ 32), and the probabilities are, as they sit in the
// accumulators, the B operand of the second product O^T[d, query] = V^T x P^T -- no exchange between lanes.
// The B operand's 16 contraction indices are matched to the accumulator rows by reading V^T's keys in the
// order (4 h + j, 8 + 4 h + j), h = lane / 32: a contraction does not care about the order of its terms as
// long as both operands agree.  K and V tiles go from memory straight into LDS, as stored ([key][d]); the A operand of the
// second product is read by the transposing LDS load (ds_read_b64_tr_b16: sixteen lanes hand in four keys of sixteen d and get four
// keys of one d each).  Against tiles moved
// through registers and transposed on the way, us: 4 prompts of up to 2048 tokens, 32 heads of 128, 149 and 132 (680 TFLOP/s); one of
// 4096 on 8 key heads 188 and 165 (830); 8 of up to 512 32.7 and 29.8; 2 of 2000 and 1500, 16 heads of 64, 47.4 and 44.4.  What
// bounds it then is the wavefronts' own instructions: reads ahead of the softmax, products in turn and priorities changed nothing.
// Bank conflicts: the 16-byte chunks of a row are permuted by an exclusive or with its
// row number, by choosing which chunk each lane of a load brings.
#include "tile_loads.h"

namespace isp {

namespace {

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kQueriesPerWave = 32;
constexpr int kWaves = 4;
constexpr int kQueryTile = kQueriesPerWave * kWaves;  // queries per workgroup
constexpr int kKeyTile = 64;

// Maximum / sum of a value with the one in the other half of the wavefront (lane ^ 32), without a trip through LDS:
// the swap leaves the lower half's value in every lane of one register and the upper half's in the other.
__device__ __forceinline__ float halves_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// x >= 0 as the sum of two halves: the upper one cut off, so that the lower one has no sign of its own, and neither is 0
// where x is not (an infinite value times either has to stay that infinity).
__device__ __forceinline__ _Float16 upper_half(float x) { return (_Float16)__builtin_amdgcn_cvt_pkrtz(x, 0.0f)[0]; }
__device__ __forceinline__ _Float16 lower_half(float x, _Float16 upper) {
    const float least = 0x1p-24f;  // fp16's smallest
    return upper_half(__builtin_amdgcn_fmed3f(x - (float)upper, least, x));
}

template <int HS>  // head size: 128, 96 or 64
__global__ __launch_bounds__(256, 2) void context_attention_f16(
    const _Float16* __restrict__ q_buf, const _Float16* __restrict__ k_cache, const _Float16* __restrict__ v_cache,
    _Float16* __restrict__ out, const int* history_length, const int* input_length, const int* context_length,
    int head_num, int kv_head_num, int max_q_len, int max_k_len, int max_seq_len, int tokens, float scale_log2e) {
    constexpr int kHeadSize = HS;
    constexpr int kDSteps = HS / 16;    // products over d per 32 x 32 block of scores
    constexpr int kDBlocks = HS / 32;   // 32-row blocks of O^T
    constexpr int kChunks = HS / 8;                      // 16-byte chunks of a key or value row
    constexpr int kRow = HS == 64 ? 8 : 16;              // and of a row in LDS: heads of 96 leave four unused
    constexpr int kLoads = kKeyTile * kRow / 256;        // of a lane per tile, of either operand
    constexpr uint32_t kTileBytes = kKeyTile * kRow * 16, kStage = 2 * kTileBytes;  // keys, then values
    // chunk c of key row r lies at c ^ key_swizzle(r), so that sixteen neighbouring rows' chunks touch every bank once; of value row
    // r at c ^ value_swizzle(r): four chunks of four neighbouring rows
    constexpr auto key_swizzle = [](int r) { return kRow == 16 ? r % 16 : r / 2 % 8; };
    constexpr auto value_swizzle = [](int r) { return kRow == 16 ? r % 4 * 4 : r / 2 % 2 * 4; };
    // Heads of 96: the probabilities as the sum of two halves, each a factor of its own product, so that they keep 21 bits (they
    // were fp32 in the kernel that served these heads before).  Scaled by 2^15 -- the sum that divides the result is, too -- so
    // that the lower halves are normal numbers down to probabilities of 2^-18.
    constexpr bool kTwoHalves = HS == 96;
    constexpr float kProbabilityExponent = kTwoHalves ? 15.0f : 0.0f;
    __shared__ __align__(1024) char tiles[2 * kStage];
    typedef __attribute__((address_space(3))) char* lds_ptr;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)tiles;

    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), half_id = lane / 32, col = lane % 32;
    // grid: x = head (fastest), y = sequence, z = query tile in DESCENDING order -- the tiles far down the causal
    // triangle visit the most key tiles, and workgroups are handed out in grid order, so the long ones start first
    // (the kernel takes as long as its longest workgroup: pinning the query tiles of a (sequence, head) pair to one
    // XCD so that they share its L2 gives up that order and measured 50 instead of 41 us)
    const int head = blockIdx.x, b = blockIdx.y, q0 = (int)(gridDim.z - 1 - blockIdx.z) * kQueryTile;
    const int len = min(read_only_i32(input_length, b), max_q_len);
    if (q0 >= len) return;  // workgroup-uniform: only padded queries here
    const int hist = read_only_i32(history_length, b);
    const int ctx = min(min(read_only_i32(context_length, b), max_k_len), max_seq_len);
    const int kv_head = head / (head_num / kv_head_num);
    const size_t kv_offset = ((size_t)b * kv_head_num + kv_head) * (size_t)max_seq_len * kHeadSize;
    const _Float16* keys = k_cache + kv_offset;
    const _Float16* values = v_cache + kv_offset;

    // keys the workgroup's last real query sees, the wavefront's last real query, this lane's query
    const int wg_visible = min(hist + min(q0 + kQueryTile, len), ctx);
    const int wave_q0 = q0 + wave * kQueriesPerWave;
    const int wave_visible = wave_q0 < len ? min(hist + min(wave_q0 + kQueriesPerWave, len), ctx) : 0;
    // keys that every query of the wavefront sees: its first query's, or none if the wavefront has padded lanes
    const int wave_all_visible = wave_q0 + kQueriesPerWave <= len ? min(hist + wave_q0 + 1, ctx) : 0;
    const int my_q = wave_q0 + col;
    const bool real = my_q < len;
    const int my_visible = real ? min(hist + my_q + 1, ctx) : 0;

    __shared__ int length_shares[kWaves];
    const int length_share = sum_lengths_thread(input_length, b);
    if (wg_visible <= 0) {  // workgroup-uniform: a context of no keys (inconsistent lengths); nothing to attend to
        sum_lengths_wave(length_share, b, length_shares);
        __syncthreads();
        const long long token = (long long)sum_lengths_total(length_shares) + my_q;
        if (real && token < tokens) {
            _Float16* o_row = out + ((size_t)token * head_num + head) * kHeadSize;
            for (int d = 8 * half_id; d < kHeadSize; d += 16) *reinterpret_cast<uint4*>(o_row + d) = make_uint4(0u, 0u, 0u, 0u);
        }
        return;
    }

    // Q^T as the B operand: lane (col, half_id) holds q[my_q][16 s + 8 half_id + 0..7] for the 8 steps over d
    half8 qf[kDSteps];
    {
        const _Float16* q_row = q_buf + (((size_t)b * head_num + head) * (size_t)max_q_len + (size_t)(real ? my_q : q0)) * kHeadSize;
#pragma unroll
        for (int s = 0; s < kDSteps; s++) {
            qf[s] = *reinterpret_cast<const half8*>(q_row + 16 * s + 8 * half_id);
            if (!real) qf[s] = half8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }

    float16v acc[kDBlocks];  // O^T[d = 32 db + rows, query = col]
#pragma unroll
    for (int db = 0; db < kDBlocks; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[db][i] = 0.0f;
    float run_max = -INFINITY, run_sum = 0.0f;

    // Two tiles are in LDS: one is computed while the loads of the other are in flight.  Rows past the visible ones re-read the last of
    // them; their scores are masked, their values cleared (a zero probability times infinity is NaN).
    uint32_t k_chunk[kLoads], v_chunk[kLoads];  // byte offsets of the chunks that this lane brings, in their rows
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        const int at = (wave * kLoads + i) * 64 + lane, r = at / kRow;
        const int kc = at % kRow ^ key_swizzle(r), vc = at % kRow ^ value_swizzle(r);
        k_chunk[i] = 16 * (kc < kChunks ? kc : kc - kChunks);
        v_chunk[i] = 16 * (vc < kChunks ? vc : vc - kChunks);
    }
    const auto load = [&](uint32_t stage_at, int kt) __attribute__((always_inline)) {
        const _Float16 *k_tile = keys + (size_t)kt * kHeadSize, *v_tile = values + (size_t)kt * kHeadSize;
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const uint32_t row = (uint32_t)min(((wave * kLoads + i) * 64 + lane) / kRow, wg_visible - 1 - kt) * (kHeadSize * 2);
            load_to_lds(stage_at + (wave * kLoads + i) * 1024, k_tile, row + k_chunk[i]);
            load_to_lds(stage_at + kTileBytes + (wave * kLoads + i) * 1024, v_tile, row + v_chunk[i]);
        }
    };
    load(lds0, 0);
    if (kKeyTile < wg_visible) load(lds0 + kStage, kKeyTile);
    sum_lengths_wave(length_share, b, length_shares);

    // where a lane reads: row col of 32 keys; of V rows 4 half_id ... of eight, four columns, for the lane that they end in
    uint32_t k_at[kDSteps], v_at[kDBlocks];
#pragma unroll
    for (int st = 0; st < kDSteps; st++) k_at[st] = lds0 + col * (kRow * 16) + 16 * ((2 * st + half_id) ^ key_swizzle(col));
#pragma unroll
    for (int db = 0; db < kDBlocks; db++) {
        const int r = 4 * half_id + lane % 16 / 4, c = 4 * db + lane / 16 % 2 * 2 + lane % 4 / 2;
        v_at[db] = lds0 + kTileBytes + r * (kRow * 16) + 16 * (c ^ value_swizzle(r)) + 8 * (lane % 2);
    }

    uint32_t stage_at = lds0;
    for (int kt = 0; kt < wg_visible; kt += kKeyTile) {
        const bool more = kt + kKeyTile < wg_visible;
        if (more) {
            wait_loads<2 * kLoads>();
        } else {
            wait_loads<0>();
#pragma unroll
            for (int i = 0; i < kLoads; i++) {
                const int at = (wave * kLoads + i) * 64 + lane;
                if (kt + at / kRow >= wg_visible) lds_clear16(stage_at + kTileBytes + at * 16);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");

        if (kt < wave_visible) {  // wavefront-uniform: tiles behind this wavefront's diagonal are skipped
            // ---- S^T[key, query] for the 64 keys: two 32-row blocks, 8 steps over d each
            // The operand reads of a block are issued together, ahead of the products that use them: read one at a
            // time, each would be waited for (an LDS round trip of a hundred cycles and more) before its product.
            float16v s[2];
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
#pragma unroll
                for (int i = 0; i < 16; i++) s[rb][i] = 0.0f;
                half8 ka[kDSteps];
#pragma unroll
                for (int st = 0; st < kDSteps; st++)
                    ka[st] = lds_read_row(k_at[st] + 32 * rb * (kRow * 16));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int st = 0; st < kDSteps; st++) s[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[st], qf[st], s[rb], 0, 0, 0);
            }
            // ---- online softmax; accumulator i of block rb is key kt + 32 rb + 8 (i / 4) + 4 half_id + i % 4
            float tile_max = -INFINITY;
            if (kt + kKeyTile > wave_all_visible) {  // wavefront-uniform: some query of this wavefront does not see the whole tile
#pragma unroll
                for (int rb = 0; rb < 2; rb++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int key = kt + 32 * rb + 8 * (i / 4) + 4 * half_id + (i % 4);
                        s[rb][i] = key < my_visible ? s[rb][i] : -INFINITY;
                    }
            }
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int i = 0; i < 16; i++) tile_max = fmaxf(tile_max, s[rb][i]);
            tile_max = halves_max(tile_max);
            const float new_max = fmaxf(run_max, tile_max);
            const float safe_max = new_max == -INFINITY ? 0.0f : new_max;  // a query with no visible key yet
            // 1 also for a column that sees no key (padded queries): its sum and accumulators are zero
            const float rescale = new_max == run_max ? 1.0f : __builtin_amdgcn_exp2f((run_max - safe_max) * scale_log2e);
            const float mc = safe_max * scale_log2e - kProbabilityExponent;
            float tile_sum = 0.0f;
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    s[rb][i] = __builtin_amdgcn_exp2f(fmaf(s[rb][i], scale_log2e, -mc));
                    tile_sum += s[rb][i];
                }
            tile_sum = halves_sum(tile_sum);
            run_sum = run_sum * rescale + tile_sum;
            run_max = new_max;
            if (__any(rescale != 1.0f)) {  // the running maximum moves in the first tiles and rarely afterwards
#pragma unroll
                for (int db = 0; db < kDBlocks; db++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[db][i] *= rescale;
            }
            // ---- O^T += V^T x P^T, 16 keys per step
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int rb = t / 2, g0 = 2 * (t % 2);
                half8 va[kDBlocks];
#pragma unroll
                for (int db = 0; db < kDBlocks; db++)
                    va[db] = __builtin_shufflevector(lds_read_transposed(v_at[db] + 16 * t * (kRow * 16)),
                                                     lds_read_transposed(v_at[db] + (16 * t + 8) * (kRow * 16)), 0, 1, 2, 3, 4, 5, 6, 7);
                half8 p, low;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float x = s[rb][4 * (g0 + e / 4) + (e % 4)];
                    p[e] = kTwoHalves ? upper_half(x) : (_Float16)x;
                    if (kTwoHalves) low[e] = lower_half(x, p[e]);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int db = 0; db < kDBlocks; db++) {
                    acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[db], p, acc[db], 0, 0, 0);
                    if (kTwoHalves) acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[db], low, acc[db], 0, 0, 0);
                }
            }
        }
        // once every wavefront has read this tile its place is free for the one after the next
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
        if (kt + 2 * kKeyTile < wg_visible) load(stage_at, kt + 2 * kKeyTile);
        const uint32_t by = stage_at == lds0 ? kStage : 0u - kStage;
        stage_at += by;
#pragma unroll
        for (int st = 0; st < kDSteps; st++) k_at[st] += by;
#pragma unroll
        for (int db = 0; db < kDBlocks; db++) v_at[db] += by;
    }

    const long long token = (long long)sum_lengths_total(length_shares) + my_q;
    // ---- O^T / sum -> the packed token row; accumulator i of block db is d = 32 db + 8 (i / 4) + 4 half_id + i % 4
    if (real && token < tokens) {
        const float inv = run_sum > 0.0f ? 1.0f / run_sum : 0.0f;
        _Float16* o_row = out + ((size_t)token * head_num + head) * kHeadSize;
#pragma unroll
        for (int db = 0; db < kDBlocks; db++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                half4 v;
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = (_Float16)(acc[db][4 * g + j] * inv);
                *reinterpret_cast<half4*>(o_row + 32 * db + 8 * g + 4 * half_id) = v;
            }
    }
}

// ---- a few queries per key / value head (a decode step): the keys and values bound the time --------------------------
//
// A workgroup serves ONE key / value head of a sequence: the queries of all heads of its group (and of all, at most a few,
// tokens) share v_mfma_f32_16x16x32_f16's 16 columns, so that a key is read once however many heads use it -- the kernel
// above would read it once per head, through a tile of 128 queries of which one is real.  A wavefront takes every
// fourth step of 32 keys, straight from memory into registers, the next step's loads in flight while it computes one:
//   S^T[key, query] = K x Q^T   lane (j = lane % 16, g = lane / 16) loads 16 bytes of key j (d = 32 i + 8 g ...): the operand as is;
//                               its results belong to query j and the keys 4 g ... 4 g + 3 of a block of 16;
//   O^T[d, query] = V^T x P^T   the contraction index is matched to that: the lane loads the kChunk elements d = kChunk j ... of
//                               its eight keys (whole rows per instruction) and transposes them in its registers, one
//                               byte-permute per dword; product c yields the rows d = kChunk (4 g + r) + c.
// The wavefronts' (maximum, sum, O) are combined through LDS; where sequences x key heads leave compute units idle, a
// sequence's keys are split over workgroups as well and a second kernel combines those.
// 16 sequences of 256-1023 keys, 32 heads (165 MB of keys and values): 41.3 us with the kernel above, 32.1 us here (5.1 TB/s); 64
// sequences of 125-500 keys, 8 key heads for 32 (85 MB): 73.3 and 17.4 us.
constexpr int kSlots = 16;     // queries (heads of the group x tokens) of a workgroup
constexpr int kStepKeys = 32;

// one workgroup's result for a query: unnormalised O, its maximum (of scale * log2 e * score) and its sum
constexpr int partial_floats(int hs) { return hs + 4; }  // + maximum, sum; padded to whole 16-byte units

typedef float float4w __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float rows_max(float x) {  // over lane % 16 == const
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return halves_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float rows_sum(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return halves_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

template <int HS, bool SPLIT>
__global__ __launch_bounds__(256, 2) void decode_attention_f16(
    const _Float16* __restrict__ q_buf, const _Float16* __restrict__ k_cache, const _Float16* __restrict__ v_cache,
    _Float16* __restrict__ out, float* __restrict__ partial, const int* history_length, const int* input_length,
    const int* context_length, int head_num, int kv_head_num, int max_q_len, int max_k_len, int max_seq_len, int tokens,
    float scale_log2e) {
    constexpr int kChunk = HS / 16, kDSteps = HS / 32, kWords = kChunk / 2;  // kWords: dwords of a lane's piece of a value row
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), j = lane % 16, g = lane / 16;
    const int kv_head = blockIdx.x, b = blockIdx.y;
    const int group = head_num / kv_head_num;
    const int len = min(read_only_i32(input_length, b), max_q_len);
    const int used = SPLIT ? group * max_q_len : group * len;  // slots with a result
    if (len <= 0) return;  // workgroup-uniform: no query row to read here, and combine_splits_f16 asks for none
    const int hist = read_only_i32(history_length, b);
    const int ctx = min(min(read_only_i32(context_length, b), max_k_len), max_seq_len);
    const int wg_visible = max(0, min(hist + len, ctx));
    const int head_in_group = j % group, my_q = j / group;
    const bool real = j < group * len;
    const int my_visible = real ? min(hist + my_q + 1, ctx) : 0;
    const size_t kv_offset = ((size_t)b * kv_head_num + kv_head) * (size_t)max_seq_len * HS;
    const _Float16 *keys = k_cache + kv_offset, *values = v_cache + kv_offset;

    half8 qf[kDSteps];
    {
        const _Float16* q_row =
            q_buf + (((size_t)b * head_num + kv_head * group + (real ? head_in_group : 0)) * (size_t)max_q_len + (real ? my_q : 0)) * HS;
#pragma unroll
        for (int i = 0; i < kDSteps; i++) {
            qf[i] = *reinterpret_cast<const half8*>(q_row + 32 * i + 8 * g);
            if (!real) qf[i] = half8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
    const int all_steps = (wg_visible + kStepKeys - 1) / kStepKeys;
    const int per_split = (all_steps + (int)gridDim.z - 1) / (int)gridDim.z;
    const int first = (int)blockIdx.z * per_split, last = min(all_steps, first + per_split);

    struct Step {
        half8 k[2][kDSteps];
        uint32_t v[8][kWords];
    } buf[2];
    auto load = [&](int which, int s) {  // a key past the visible ones re-reads the last visible row: masked (blanked) below
        Step& t = buf[which];
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            const _Float16* row = keys + (size_t)min(s * kStepKeys + 16 * blk + j, wg_visible - 1) * HS + 8 * g;
#pragma unroll
            for (int i = 0; i < kDSteps; i++) t.k[blk][i] = *reinterpret_cast<const half8*>(row + 32 * i);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const _Float16* row = values + (size_t)min(s * kStepKeys + 16 * (i / 4) + 4 * g + i % 4, wg_visible - 1) * HS + kChunk * j;
            if constexpr (kWords == 4) {
                const uint4 x = *reinterpret_cast<const uint4*>(row);
                t.v[i][0] = x.x, t.v[i][1] = x.y, t.v[i][2] = x.z, t.v[i][3] = x.w;
            } else {
                const uint2 x = *reinterpret_cast<const uint2*>(row);
                t.v[i][0] = x.x, t.v[i][1] = x.y;
            }
        }
    };
    float4w acc[kChunk];
#pragma unroll
    for (int c = 0; c < kChunk; c++) acc[c] = float4w{0.0f, 0.0f, 0.0f, 0.0f};
    float run_max = -INFINITY, run_sum = 0.0f;  // run_sum: this lane's keys only
    auto compute = [&](int which, int s) {
        const Step& t = buf[which];
        float4w sc[2];
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            sc[blk] = float4w{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < kDSteps; i++) sc[blk] = __builtin_amdgcn_mfma_f32_16x16x32_f16(t.k[blk][i], qf[i], sc[blk], 0, 0, 0);
        }
        float m = -INFINITY;
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = s * kStepKeys + 16 * blk + 4 * g + r;
                sc[blk][r] = key < my_visible ? sc[blk][r] * scale_log2e : -INFINITY;
                m = fmaxf(m, sc[blk][r]);
            }
        const float new_max = fmaxf(run_max, rows_max(m));
        const float safe_max = new_max == -INFINITY ? 0.0f : new_max;  // no visible key yet
        // 1 also for a column without a query: its sum and accumulators are zero
        const float rescale = new_max == run_max ? 1.0f : __builtin_amdgcn_exp2f(run_max - safe_max);
        run_max = new_max;
        run_sum *= rescale;
        half8 p;
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float e = __builtin_amdgcn_exp2f(sc[blk][r] - safe_max);
                run_sum += e;
                p[4 * blk + r] = (_Float16)e;
            }
        if (__any(rescale != 1.0f)) {
#pragma unroll
            for (int c = 0; c < kChunk; c++) acc[c] *= rescale;
        }
#pragma unroll
        for (int c = 0; c < kChunk; c++) {
            union { uint32_t u[4]; half8 h; } vt;
#pragma unroll
            for (int i = 0; i < 4; i++)
                vt.u[i] = __builtin_amdgcn_perm(t.v[2 * i + 1][c / 2], t.v[2 * i][c / 2], c % 2 ? 0x07060302u : 0x05040100u);
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vt.h, p, acc[c], 0, 0, 0);
        }
    };
    // the only step with keys past the visible ones is the last of all, which its wavefront takes last: their value rows count as
    // zero (0 x inf is NaN)
    auto blank = [&](int which, int s) {
        if ((s + 1) * kStepKeys <= wg_visible) return;  // wavefront-uniform
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t keep = s * kStepKeys + 16 * (i / 4) + 4 * g + i % 4 < wg_visible ? 0xffffffffu : 0u;
#pragma unroll
            for (int w = 0; w < kWords; w++) buf[which].v[i][w] &= keep;
        }
    };
    int s = first + wave;
    if (s < last) {
        load(0, s);
        for (;;) {
            if (s + kWaves >= last) {
                blank(0, s);
                compute(0, s);
                break;
            }
            load(1, s + kWaves);
            compute(0, s);
            s += kWaves;
            if (s + kWaves >= last) {
                blank(1, s);
                compute(1, s);
                break;
            }
            load(0, s + kWaves);
            compute(1, s);
            s += kWaves;
        }
    }

    __shared__ __align__(16) float o_lds[kWaves][kSlots][HS];
    __shared__ float m_lds[kWaves][kSlots], l_lds[kWaves][kSlots];
    run_sum = rows_sum(run_sum);
    if (g == 0) {
        m_lds[wave][j] = run_max;
        l_lds[wave][j] = run_sum;
    }
    if (j < used) {
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int c = 0; c < kChunk; c += 4)
                *reinterpret_cast<float4w*>(&o_lds[wave][j][kChunk * (4 * g + r) + c]) =
                    float4w{acc[c][r], acc[c + 1][r], acc[c + 2][r], acc[c + 3][r]};
    }
    __shared__ int length_shares[kWaves];
    if (!SPLIT) sum_lengths_wave(sum_lengths_thread(input_length, b), b, length_shares);
    __syncthreads();
    const int first_token = SPLIT ? 0 : sum_lengths_total(length_shares);
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
        const int head = kv_head * group + slot % group, q = slot / group;
        if (SPLIT) {
            float* p = partial + ((((size_t)b * head_num + head) * max_q_len + q) * gridDim.z + blockIdx.z) * partial_floats(HS);
            *reinterpret_cast<float4w*>(p + d) = o;
            if (d == 0) p[HS] = m, p[HS + 1] = l;
        } else {
            const long long token = (long long)first_token + q;
            if (token < tokens) {
                const float inv = l > 0.0f ? 1.0f / l : 0.0f;
                half4 h;
#pragma unroll
                for (int e = 0; e < 4; e++) h[e] = (_Float16)(o[e] * inv);
                *reinterpret_cast<half4*>(out + ((size_t)token * head_num + head) * HS + d) = h;
            }
        }
    }
}

// The splits of a query together: a wavefront per (head, sequence and token), HS / 64 elements per lane.
template <int HS>
__global__ __launch_bounds__(64) void combine_splits_f16(const float* __restrict__ partial, _Float16* __restrict__ out,
                                                         const int* input_length, int head_num, int max_q_len, int splits,
                                                         int tokens) {
    const int lane = threadIdx.x, head = blockIdx.x, b = (int)blockIdx.y / max_q_len, q = (int)blockIdx.y % max_q_len;
    if (q >= read_only_i32(input_length, b)) return;  // workgroup-uniform: no such query
    int n = 0;
    for (int i = lane; i < b; i += 64) n += read_only_i32(input_length, i);
    const float* p = partial + (((size_t)b * head_num + head) * max_q_len + q) * (size_t)splits * partial_floats(HS);
    float m = -INFINITY, l = 0.0f;
    for (int z = lane; z < splits; z += 64) m = fmaxf(m, p[z * partial_floats(HS) + HS]);
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off, 64));
        n += __shfl_xor(n, off, 64);
    }
    const float safe = m == -INFINITY ? 0.0f : m;
    float o[HS / 64] = {};
    constexpr int kAtOnce = 8;  // splits whose loads are on their way together; those past the last re-read it
    for (int z0 = 0; z0 < splits; z0 += kAtOnce) {
        float part[kAtOnce][HS / 64 + 2];
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            const float* pz = p + min(z0 + i, splits - 1) * partial_floats(HS);
            part[i][0] = pz[HS];
            part[i][1] = pz[HS + 1];
#pragma unroll
            for (int d = 0; d < HS / 64; d++) part[i][2 + d] = pz[HS / 64 * lane + d];
        }
#pragma unroll
        for (int i = 0; i < kAtOnce; i++)
#pragma unroll
            for (int d = 0; d < HS / 64 + 2; d++) asm volatile("" : "+v"(part[i][d]));  // or the loads move behind the test below
#pragma unroll
        for (int i = 0; i < kAtOnce; i++) {
            if (z0 + i >= splits) break;  // uniform
            const float e = __builtin_amdgcn_exp2f(part[i][0] - safe);
            l += e * part[i][1];
#pragma unroll
            for (int d = 0; d < HS / 64; d++) o[d] += e * part[i][2 + d];
        }
    }
    const long long token = (long long)n + q;
    if (token >= tokens) return;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int i = 0; i < HS / 64; i++) out[((size_t)token * head_num + head) * HS + HS / 64 * lane + i] = (_Float16)(o[i] * inv);
}

}  // namespace

// Workgroups that share a (sequence, key head): enough for two on every compute unit, each with at least 128 keys (four
// steps, one per wavefront).  One where the second kernel's grid, with a row per sequence and query, would not hold them.
static int attention_splits(int batch, int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len) {
    if (batch <= 0 || kv_head_num <= 0 || head_size == 96 || head_num / kv_head_num * (long long)max_q_len > kSlots ||
        (long long)batch * max_q_len > 65535)
        return 1;
    const long long groups = (long long)batch * kv_head_num, units = resident_waves() / 32;
    long long splits = (2 * units) / groups;
    const long long most = (max_k_len + 4 * kStepKeys - 1) / (4 * kStepKeys);
    if (splits > most) splits = most;
    return splits < 1 ? 1 : (int)splits;
}

size_t attention_workspace(int batch, int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len) {
    const int splits = attention_splits(batch, head_num, kv_head_num, head_size, max_q_len, max_k_len);
    return splits == 1 ? 0 : (size_t)splits * batch * head_num * max_q_len * partial_floats(head_size) * sizeof(float);
}

// csrc/context_attention_f32.hip: fp16 heads of 96 elements, computed in fp32
int context_attention_f16_96(const __half* q, const __half* k_cache, const __half* v_cache, __half* out,
                             const int32_t* history_length, const int32_t* input_length, const int32_t* context_length, int layer,
                             int batch, int head_num, int kv_head_num, int max_q_len, int max_k_len, int max_seq_len,
                             int token_num, float scale, hipStream_t stream);

// Heads of 96 elements have two kernels.  The fp32 one has 16 queries per workgroup, whose four wavefronts split a sequence's keys; it
// serves up to 16 queries, and more while its workgroups all run at once.  Beyond that the matrix rate counts, and the
// tiled one here has four to five times its.  500 ... 8000 keys, at most one workgroup per compute unit: 17 ... 216 against 23 ... 254
// us; at 384 workgroups 27 ... 305 against 23 ... 254; 2 x 2048 tokens with 32 heads 535 against 113 (the padded form: 379).  256
// sequences, 32 heads, 8 and 16 queries on 50 keys 58 and 75 against 88 and 121, 20 queries 134 against 122.
static bool attention_96_in_fp32(int batch, int head_num, int max_q_len) {
    return max_q_len <= 16 || (long long)batch * head_num * ((max_q_len + 15) / 16) <= resident_waves() / 32;
}

// `workspace` NULL: a sequence's keys are not split.
int context_attention(const _Float16* q, const _Float16* k_cache, const _Float16* v_cache, _Float16* out,
                      const int32_t* history_length, const int32_t* input_length, const int32_t* context_length,
                      int layer, int batch, int head_num, int kv_head_num, int head_size, int max_q_len,
                      int max_k_len, int max_seq_len, int token_num, float scale, float* workspace, hipStream_t stream) {
    if (layer < 0 || batch < 0 || head_num <= 0 || kv_head_num <= 0 || head_num % kv_head_num != 0 || max_q_len < 0 ||
        max_k_len < 0 || max_seq_len < 0 || token_num < 0 || !(scale > 0.0f))
        return ISP_ERR_BAD_SHAPE;
    if (head_size == 96 && attention_96_in_fp32(batch, head_num, max_q_len))
        return context_attention_f16_96(reinterpret_cast<const __half*>(q), reinterpret_cast<const __half*>(k_cache),
                                        reinterpret_cast<const __half*>(v_cache), reinterpret_cast<__half*>(out), history_length,
                                        input_length, context_length, layer, batch, head_num, kv_head_num, max_q_len, max_k_len,
                                        max_seq_len, token_num, scale, stream);
    if (head_size != 128 && head_size != 96 && head_size != 64) return ISP_ERR_UNSUPPORTED;
    if (batch == 0 || max_q_len == 0 || token_num == 0) return ISP_OK;
    if (max_k_len == 0 || max_seq_len == 0) return ISP_ERR_BAD_SHAPE;
    const int tiles = (max_q_len + kQueryTile - 1) / kQueryTile;
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
    const float scale_log2e = scale * 1.4426950408889634f;
    if ((long long)(head_num / kv_head_num) * max_q_len <= kSlots) {
        if (!aligned16(workspace)) return ISP_ERR_UNSUPPORTED;
        const int splits = workspace ? attention_splits(batch, head_num, kv_head_num, head_size, max_q_len, max_k_len) : 1;
        const dim3 grid((unsigned)kv_head_num, (unsigned)batch, (unsigned)splits);
#define ISP_LAUNCH_DECODE(HS, SPLIT)                                                                                          \
    hipLaunchKernelGGL((decode_attention_f16<HS, SPLIT>), grid, dim3(256), 0, stream, q, k_cache + slice, v_cache + slice, out, \
                       workspace, history_length, input_length, context_length, head_num, kv_head_num, max_q_len, max_k_len,  \
                       max_seq_len, token_num, scale_log2e)
        if (splits == 1) {
            if (head_size == 128) ISP_LAUNCH_DECODE(128, false);
            else ISP_LAUNCH_DECODE(64, false);
            return note_launch(hipGetLastError());
        }
        if (head_size == 128) ISP_LAUNCH_DECODE(128, true);
        else ISP_LAUNCH_DECODE(64, true);
#undef ISP_LAUNCH_DECODE
        const int status = note_launch(hipGetLastError());
        if (status != ISP_OK) return status;
        const dim3 queries((unsigned)head_num, (unsigned)(batch * max_q_len));
        if (head_size == 128)
            hipLaunchKernelGGL(combine_splits_f16<128>, queries, dim3(64), 0, stream, workspace, out, input_length, head_num,
                               max_q_len, splits, token_num);
        else
            hipLaunchKernelGGL(combine_splits_f16<64>, queries, dim3(64), 0, stream, workspace, out, input_length, head_num,
                               max_q_len, splits, token_num);
        return note_launch(hipGetLastError());
    }
    const dim3 grid((unsigned)head_num, (unsigned)batch, (unsigned)tiles);
#define ISP_LAUNCH_ATTENTION(HS)                                                                                    \
    hipLaunchKernelGGL(context_attention_f16<HS>, grid, dim3(256), 0, stream, q, k_cache + slice, v_cache + slice, out, \
                       history_length, input_length, context_length, head_num, kv_head_num, max_q_len, max_k_len,   \
                       max_seq_len, token_num, scale_log2e)
    if (head_size == 128) ISP_LAUNCH_ATTENTION(128);
    else if (head_size == 96) ISP_LAUNCH_ATTENTION(96);
    else ISP_LAUNCH_ATTENTION(64);
#undef ISP_LAUNCH_ATTENTION
    return note_launch(hipGetLastError());
}

}  // namespace isp

extern "C" {

size_t isp_context_attention_f16_workspace(int batch, int head_num, int kv_head_num, int head_size, int max_q_len,
                                           int max_k_len) {
    return isp::attention_workspace(batch, head_num, kv_head_num, head_size, max_q_len, max_k_len);
}

int isp_context_attention_split_f16(const void* q, const void* k_cache, const void* v_cache, void* out,
                                    const int32_t* history_length, const int32_t* input_length,
                                    const int32_t* context_length, int layer, int batch, int head_num, int kv_head_num,
                                    int head_size, int max_q_len, int max_k_len, int max_seq_len, int token_num, float scale,
                                    void* workspace, isp_stream_t stream) {
    return isp::context_attention(static_cast<const _Float16*>(q), static_cast<const _Float16*>(k_cache),
                                  static_cast<const _Float16*>(v_cache), static_cast<_Float16*>(out), history_length,
                                  input_length, context_length, layer, batch, head_num, kv_head_num, head_size, max_q_len,
                                  max_k_len, max_seq_len, token_num, scale, static_cast<float*>(workspace),
                                  static_cast<hipStream_t>(stream));
}

int isp_context_attention_f16(const void* q, const void* k_cache, const void* v_cache, void* out,
                              const int32_t* history_length, const int32_t* input_length, const int32_t* context_length,
                              int layer, int batch, int head_num, int kv_head_num, int head_size, int max_q_len,
                              int max_k_len, int max_seq_len, int token_num, float scale, isp_stream_t stream) {
    return isp_context_attention_split_f16(q, k_cache, v_cache, out, history_length, input_length, context_length, layer,
                                           batch, head_num, kv_head_num, head_size, max_q_len, max_k_len, max_seq_len,
                                           token_num, scale, nullptr, stream);
}

}  // extern "C"
