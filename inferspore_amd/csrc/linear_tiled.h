// Product of a layer with more rows than the skinny kernel (linear_rows.h) is made for: C[m, n] = A[m, k] x W[k, n], fp16, row-major,
// fp32 accumulation, weights read as they lie in memory.
//
// A workgroup owns a BM x BN tile and walks k in steps of 64.  The operands of a step go from memory straight into LDS
// (global_load_lds, 16 bytes per lane, no registers in between), STAGES steps deep.  Matrix cores (v_mfma_f32_16x16x32_f16) want
// eight consecutive k per lane from both operands: rows of A are that already (ds_read_b128), columns of W are read by the transposing
// LDS load (ds_read_b64_tr_b16: sixteen lanes hand in four rows of sixteen columns and get one column each).  The product is
// formed transposed, W^T x A^T, so that a lane ends with neighbouring columns of one output row.
//
// Bank conflicts: LDS rows are whole powers of two, so the 16-byte chunks of a row are permuted by an exclusive or with its row number -- by
// choosing which chunk each lane of a load brings, as the loads fill LDS in lane order.  Chunk c of row r of A lies at c ^ (r / 2 % 8),
// of W at c ^ swizzle(r); sixteen (A) and thirty-two (W) lanes then touch every bank once.
//
// Order of a step, per wavefront: the operands of the next 32 k are read while the products of these are computed, one read behind
// every second product, and once the last are in registers (one barrier per step) the freed buffer is loaded again, one load
// behind every few products.  The order is pinned (sched_barrier): left to itself the compiler reads each operand right before its
// product, 1070 against 940 us at 6460 x 4096 x 22016.  The products' issue slots are 58 % used there and the clock is down at 1.7 to 1.9
// GHz: the chip's power is the limit, and the tile that moves the fewest bytes through LDS is the best one.
//
// Against the library's product of the same operands (hipBLASLt), us: 64 x 4096 x 4096 27, 10.7; 128 x 11008 x 4096 95, 25; 462 x 4096 x
// 12288 66, 54; 462 x 11008 x 4096 98, 49; 660 x 1024 x 3072 17.5, 11.2; 2610 x 4096 x 22016 487, 411; 6460 x 4096 x 22016 1062, 940.
#pragma once

#include "tile_loads.h"

namespace isp {

// What becomes of the sums: fp16 to `out`; fp32 to partial[split], for the consumer to add up; or, with W's columns [0, n / 2) gates and
// [n / 2, n) up projections, SwiGLU of the two products rounded to fp16 -- what the separate kernel computes from the stored product, same
// bits -- to `out` [m, n / 2].
enum TiledResult { kTiledHalf = 0, kTiledPartial = 1, kTiledSwiglu = 2 };

constexpr int kTiledStep = 64;  // k per step

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int RESULT>
__global__ __launch_bounds__(kWave* WAVES_M* WAVES_N, 2) void linear_tiled_f16(const __half* __restrict__ a, const __half* __restrict__ w,
                                                                               __half* __restrict__ out, float* __restrict__ partial,
                                                                               int m, int n, int k, int steps_per_split) {
    constexpr int WAVES = WAVES_M * WAVES_N, TM = BM / WAVES_M, TN = BN / WAVES_N;  // a wavefront's part of the tile
    constexpr int MI = TM / 16, NI = TN / 16, SUB = kTiledStep / 32;
    constexpr int CA = kTiledStep / 8, CW = BN / 8;                                                    // chunks of a row
    constexpr int LA = BM * CA / (kWave * WAVES), LW = kTiledStep * CW / (kWave * WAVES), LOADS = LA + LW;  // loads of a wavefront per step
    constexpr uint32_t kABytes = BM * kTiledStep * 2, kStage = kABytes + kTiledStep * BN * 2;
    static_assert(LA * kWave * WAVES == BM * CA && LW * kWave * WAVES == kTiledStep * CW && CW % 8 == 0 && NI % 2 == 0, "whole loads and pairs");
    static_assert(STAGES * kStage <= 160 * 1024, "LDS");
    // SwiGLU: the tile's columns alternate between gates and up projections, kGroup chunks at a time, so that a wavefront holds both
    constexpr int kGroup = TN % 64 == 0 ? 4 : 2;
    __shared__ __align__(1024) char lds_bytes[STAGES * kStage];
    typedef __attribute__((address_space(3))) char* lds_ptr;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds_bytes;

    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), j = lane % 16, g = lane / 16;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;

    const int cols = RESULT == kTiledSwiglu ? BN / 2 : BN, width = RESULT == kTiledSwiglu ? n / 2 : n;  // result columns
    const TilePlace place = place_tile((m + BM - 1) / BM, (width + cols - 1) / cols);
    const int m0 = place.row * BM, n0 = place.col * cols;

    const int steps = (k + kTiledStep - 1) / kTiledStep;
    const int first = (int)blockIdx.y * steps_per_split, last = min(steps, first + steps_per_split), count = last - first;
    // a last step that is not whole is taken first: its loads and the clearing of what is past k then stay out of the loop
    const bool ragged = last == steps && k % kTiledStep != 0;

    // Where a lane's loads come from.  Rows past m and columns past n re-read the last ones; their results are not stored.
    constexpr auto w_swizzle = [](int r) { return (CW % 16 == 0 ? r % 4 * 4 : r / 2 % 2 * 4) | r / 8 % 2 * 2; };
    uint32_t a_off[LA], w_off[LW];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int at = (wave * LA + i) * kWave + lane, r = at / CA, c = at % CA ^ r / 2 % 8;
        a_off[i] = ((uint32_t)(min(m0 + r, m - 1) - m0) * (uint32_t)k + 8u * c) * 2u;
    }
#pragma unroll
    for (int i = 0; i < LW; i++) {
        const int at = (wave * LW + i) * kWave + lane, r = at / CW, c = at % CW ^ w_swizzle(r);
        int col = min(n0 + 8 * c, width - 8);
        if (RESULT == kTiledSwiglu) col = min(n0 + 8 * (c % kGroup + c / (2 * kGroup) * kGroup), width - 8) + c / kGroup % 2 * width;
        w_off[i] = ((uint32_t)r * (uint32_t)n + (uint32_t)col) * 2u;
    }
    const char* a_next = reinterpret_cast<const char*>(a + (size_t)m0 * (size_t)k + (size_t)first * kTiledStep);
    const char* w_next = reinterpret_cast<const char*>(w + (size_t)first * kTiledStep * (size_t)n);
    const size_t w_step = (size_t)kTiledStep * (size_t)n * 2u;
    const auto load = [&](auto i_, uint32_t stage_at) __attribute__((always_inline)) {  // load i of LOADS
        constexpr int i = decltype(i_)::value;
        if constexpr (i < LA) load_to_lds(stage_at + (wave * LA + i) * 1024, a_next, a_off[i]);
        else load_to_lds(stage_at + kABytes + (wave * LW + i - LA) * 1024, w_next, w_off[i - LA]);
    };
    const auto advance = [&]() __attribute__((always_inline)) {
        a_next += kTiledStep * 2;
        w_next += w_step;
    };

    // Where a lane reads: rows j of A's blocks, chunk 4 sub + g; of W lane (e, c) of each sixteen hands in row e, columns 4 c ... of
    // the four rows that its sixteen lanes need.
    uint32_t a_at[SUB], w_at[NI];
#pragma unroll
    for (int s = 0; s < SUB; s++) a_at[s] = lds0 + (wm * TM + j) * (kTiledStep * 2) + 16 * ((4 * s + g) ^ j / 2 % 8);
#pragma unroll
    for (int y = 0; y < NI; y++) {
        const int r = 8 * g + lane % 16 / 4, col = wn * TN + 16 * y + 4 * (lane % 4);
        w_at[y] = lds0 + kABytes + r * (BN * 2) + 16 * (col / 8 ^ w_swizzle(r)) + 2 * (col % 8);
    }

    float4v acc[MI][NI];
#pragma unroll
    for (int x = 0; x < MI; x++)
#pragma unroll
        for (int y = 0; y < NI; y++) acc[x][y] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    half8 a_reg[2][MI], w_reg[2][NI];
    half4 w_low;
    constexpr int READS = MI + 2 * NI, PRODUCTS = MI * NI;
    // read i of READS: the first column block, the rows, the other column blocks -- the order in which the products want them
    const auto read = [&](auto set_, auto sub_, auto i_) __attribute__((always_inline)) {
        constexpr int set = decltype(set_)::value, sub = decltype(sub_)::value, i = decltype(i_)::value;
        if constexpr (i >= 2 && i < 2 + MI) {
            a_reg[set][i - 2] = lds_read_row(a_at[sub] + (i - 2) * 16 * kTiledStep * 2);
        } else {
            constexpr int y = i < 2 ? 0 : (i - MI) / 2, half = i < 2 ? i : (i - MI) % 2;
            const half4 v = lds_read_transposed(w_at[y] + (32 * sub + 4 * half) * BN * 2);
            if constexpr (half == 0) w_low = v;
            else w_reg[set][y] = __builtin_shufflevector(w_low, v, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    // the products of one set of operands; behind them the reads of the other set, over the first three quarters of them, and the loads
    const auto products = [&](auto set_, auto next_sub_, auto load_, uint32_t load_at) __attribute__((always_inline)) {
        constexpr int set = decltype(set_)::value;
        constexpr int read_span = PRODUCTS * 3 / 4 > 0 ? PRODUCTS * 3 / 4 : 1;
        static_for<PRODUCTS>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            acc[i % MI][i / MI] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w_reg[set][i / MI], a_reg[set][i % MI], acc[i % MI][i / MI], 0, 0, 0);
            constexpr int r0 = (i * READS + read_span - 1) / read_span, r1 = ((i + 1) * READS + read_span - 1) / read_span;
            static_for<(r1 < READS ? r1 : READS) - (r0 < READS ? r0 : READS)>([&](auto d) __attribute__((always_inline)) {
                read(std::integral_constant<int, 1 - set>{}, next_sub_, std::integral_constant<int, r0 + decltype(d)::value>{});
            });
            if constexpr (decltype(load_)::value) {
                constexpr int l0 = (i * LOADS + PRODUCTS - 1) / PRODUCTS, l1 = ((i + 1) * LOADS + PRODUCTS - 1) / PRODUCTS;
                static_for<l1 - l0>([&](auto d) __attribute__((always_inline)) {
                    load(std::integral_constant<int, l0 + decltype(d)::value>{}, load_at);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (decltype(load_)::value) advance();
    };

    // ---- the first steps' loads
    if (ragged) {  // the last step: what lies past k re-reads the last chunk (row) that exists
        const int k0 = (steps - 1) * kTiledStep;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int at = (wave * LA + i) * kWave + lane, r = at / CA, c = at % CA ^ r / 2 % 8, past = max(0, k0 + 8 * c - (k - 8));
            load_to_lds(lds0 + (wave * LA + i) * 1024, a + (size_t)m0 * (size_t)k + k0, a_off[i] - 2u * past);
        }
#pragma unroll
        for (int i = 0; i < LW; i++) {
            const int at = (wave * LW + i) * kWave + lane, r = at / CW, past = max(0, k0 + r - (k - 1));
            load_to_lds(lds0 + kABytes + (wave * LW + i) * 1024, w + (size_t)k0 * (size_t)n, w_off[i] - 2u * past * (uint32_t)n);
        }
    }
#pragma unroll
    for (int s = 0; s < STAGES; s++) {
        if ((s > 0 || !ragged) && s < count) {
            static_for<LOADS>([&](auto i) __attribute__((always_inline)) { load(i, lds0 + s * kStage); });
            advance();
        }
    }
    if (count >= STAGES) wait_loads<(STAGES - 1) * LOADS>();
    else wait_loads<0>();
    if (ragged) {  // every lane clears what it has brought from past k, on both sides (0 x inf is NaN)
        const int k0 = (steps - 1) * kTiledStep;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int at = (wave * LA + i) * kWave + lane, r = at / CA, c = at % CA ^ r / 2 % 8;
            if (k0 + 8 * c >= k) lds_clear16(lds0 + at * 16);
        }
#pragma unroll
        for (int i = 0; i < LW; i++) {
            const int at = (wave * LW + i) * kWave + lane, r = at / CW;
            if (k0 + r >= k) lds_clear16(lds0 + kABytes + at * 16);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
    constexpr std::integral_constant<int, 0> zero{};
    static_for<READS>([&](auto i) __attribute__((always_inline)) { read(zero, zero, i); });

    // ---- a step; `more`: the loads of the step after the next are in flight as well
    static_assert(SUB == 2, "two sets of operands per step");
    int stage = 0;
    const auto step = [&](bool more, auto load_) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 1> one{};
        products(zero, one, std::false_type{}, 0);
        // the operands of this step are all in registers: once every wavefront is here, its buffer is free and the next step's full
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        if (more) wait_loads<(STAGES - 2) * LOADS>();
        else wait_loads<0>();
        asm volatile("s_barrier" : : : "memory");
        const uint32_t freed = lds0 + stage * kStage;
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        const uint32_t by = stage == 0 ? 0u - (STAGES - 1) * kStage : kStage;
#pragma unroll
        for (int s = 0; s < SUB; s++) a_at[s] += by;
#pragma unroll
        for (int y = 0; y < NI; y++) w_at[y] += by;
        products(one, zero, load_, freed);  // behind the last step it reads what lies in the next buffer, for nobody
    };
    int t = 0;
#pragma unroll 1
    for (; t + STAGES < count; t++) step(true, std::true_type{});
#pragma unroll 1
    for (; t < count; t++) step(t + STAGES == count, std::false_type{});

    // ---- lane (j, g) holds row j and columns 4 g ... 4 g + 3 of every block.  Two blocks exchanged between neighbouring g leave eight
    //      neighbouring columns, 16 (g % 2) + 8 (g / 2) of the two blocks' 32
    constexpr bool kPairs = RESULT != kTiledSwiglu || kGroup == 4;
    if constexpr (kPairs) {
#pragma unroll
        for (int x = 0; x < MI; x++)
#pragma unroll
            for (int y = 0; y < NI; y += 2)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[x][y][e]), __float_as_uint(acc[x][y + 1][e]), false, false);
                    acc[x][y][e] = __uint_as_float(s[0]);
                    acc[x][y + 1][e] = __uint_as_float(s[1]);
                }
    }
    const auto swiglu = [](float gate, float up) {
        const float a16 = __half2float(Elem<__half>::from_f32(gate)), b16 = __half2float(Elem<__half>::from_f32(up));
        return silu_for<__half>(a16) * b16;
    };
#pragma unroll
    for (int x = 0; x < MI; x++) {
        const int row = m0 + wm * TM + 16 * x + j;
        if (row >= m) continue;
        if constexpr (!kPairs) {
#pragma unroll
            for (int y = 0; y < NI; y += 2) {
                const int col = n0 + wn * TN / 2 + 8 * y + 4 * g;
                float f[4];
#pragma unroll
                for (int e = 0; e < 4; e++) f[e] = Elem<__half>::pinned(swiglu(acc[x][y][e], acc[x][y + 1][e]));
                const __half2 lo = __floats2half2_rn(f[0], f[1]), hi = __floats2half2_rn(f[2], f[3]);
                if (col < width)
                    *reinterpret_cast<uint2*>(out + (size_t)row * (size_t)width + col) =
                        make_uint2(*reinterpret_cast<const uint32_t*>(&lo), *reinterpret_cast<const uint32_t*>(&hi));
            }
            continue;
        }
#pragma unroll
        for (int y = 0; y < NI; y += RESULT == kTiledSwiglu ? 4 : 2) {
            const int col = n0 + (RESULT == kTiledSwiglu ? wn * TN / 2 + 8 * y : wn * TN + 16 * y) + 16 * (g % 2) + 8 * (g / 2);
            if (col >= width) continue;  // width is a multiple of 8: eight columns exist together
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                f[e] = acc[x][y + e / 4][e % 4];
                if (RESULT == kTiledSwiglu) f[e] = swiglu(f[e], acc[x][(y + 2 + e / 4) % NI][e % 4]);
            }
            const size_t at = (size_t)row * (size_t)width + col;
            if (RESULT == kTiledPartial) {
                float* p = partial + (size_t)blockIdx.y * (size_t)m * (size_t)n + at;
                *reinterpret_cast<float4v*>(p) = float4v{f[0], f[1], f[2], f[3]};
                *reinterpret_cast<float4v*>(p + 4) = float4v{f[4], f[5], f[6], f[7]};
            } else {
                store16(out + at, Elem<__half>::pack(f));
            }
        }
    }
}

}  // namespace isp
