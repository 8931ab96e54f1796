// Product of a layer in fp32: C[m, n] = A[m, k] x W[k, n], row-major, fp32 products and sums, weights read as they lie in memory.
//
// A workgroup owns a BM x BN tile and walks k in steps of 32, operands straight from memory into LDS, STAGES steps deep, as the fp16
// kernel does (linear_tiled.h).  Matrix cores (v_mfma_f32_16x16x4_f32: lane (j, g) brings row j of A and column j of W at one k) do not
// care which four k meet in one product, so lane (j, g) reads four consecutive k of its row of A at once (k = 4 g + e of sixteen) and
// takes them in turn, e = 0 ... 3; and not which columns of W make up a block, so it reads NI consecutive columns of row 4 g + e, one
// for each of NI blocks: column NI j + y for block y.  A lane then ends with NI neighbouring columns of its output rows.
//
// Sums: a lane keeps two for every value, of the even and of the odd sixteens of k.  With one, sums of few rows, which the library splits
// further, were up to 1.38 times as far from 64 bits as the library's.
//
// Bank conflicts: rows of A are 128 bytes and their 16-byte chunk c lies at c ^ (r / 2 % 8), so that sixteen lanes of a read touch every
// bank once; rows of W are whole multiples of 256 bytes, and where lanes read less than 16 bytes of them, the rows of different g are moved
// apart by an exclusive or likewise (w_swizzle).
#pragma once

#include "tile_loads.h"

namespace isp {

constexpr int kTiledStepF32 = 32;  // k per step

// Sums of steps [blockIdx.y * steps_per_split, ...) to out[blockIdx.y][m][n]; or, with W's columns [0, n / 2) gates and [n / 2, n) up
// projections, SwiGLU of the two products -- what the separate kernel computes from the stored product, same bits -- to out [m, n / 2].
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool SWIGLU>
__global__ __launch_bounds__(kWave* WAVES_M* WAVES_N, 2) void linear_tiled_f32(const float* __restrict__ a, const float* __restrict__ w,
                                                                               float* __restrict__ out, int m, int n, int k,
                                                                               int steps_per_split) {
    constexpr int WAVES = WAVES_M * WAVES_N, TM = BM / WAVES_M, TN = BN / WAVES_N;  // a wavefront's part of the tile
    constexpr int MI = TM / 16, NI = TN / 16, SUB = kTiledStepF32 / 16;
    constexpr int CA = kTiledStepF32 / 4, CW = BN / 4;                                                         // chunks of a row
    constexpr int LA = BM * CA / (kWave * WAVES), LW = kTiledStepF32 * CW / (kWave * WAVES), LOADS = LA + LW;  // loads of a wavefront per step
    constexpr uint32_t kABytes = BM * kTiledStepF32 * 4, kStage = kABytes + kTiledStepF32 * BN * 4;
    static_assert(LA * kWave * WAVES == BM * CA && LW * kWave * WAVES == kTiledStepF32 * CW && CW % 16 == 0, "whole loads");
    static_assert(MI * 16 * WAVES_M == BM && NI * 16 * WAVES_N == BN && (NI == 1 || NI == 2 || NI == 4), "whole blocks");
    static_assert(STAGES * kStage <= 160 * 1024, "LDS");
    __shared__ __align__(1024) char lds_bytes[STAGES * kStage];
    typedef __attribute__((address_space(3))) char* lds_ptr;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)lds_bytes;

    const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), j = lane % 16, g = lane / 16;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int result_cols = SWIGLU ? BN / 2 : BN, width = SWIGLU ? n / 2 : n;
    const TilePlace place = place_tile((m + BM - 1) / BM, (width + result_cols - 1) / result_cols);
    const int m0 = place.row * BM, n0 = place.col * result_cols;

    const int steps = (k + kTiledStepF32 - 1) / kTiledStepF32;
    const int first = (int)blockIdx.y * steps_per_split, last = min(steps, first + steps_per_split), count = last - first;
    // a last step that is not whole is taken first: its loads and the clearing of what is past k then stay out of the loop
    const bool ragged = last == steps && k % kTiledStepF32 != 0;

    // Where a lane's loads come from.  Rows past m and columns past n re-read the last ones; their results are not stored.
    constexpr auto w_swizzle = [](int r) { return NI == 4 ? 0 : NI == 2 ? r / 4 % 2 * 8 : r / 4 % 4 * 4; };
    uint32_t a_off[LA], w_off[LW];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int at = (wave * LA + i) * kWave + lane, r = at / CA, c = at % CA ^ r / 2 % 8;
        a_off[i] = ((uint32_t)(min(m0 + r, m - 1) - m0) * (uint32_t)k + 4u * c) * 4u;
    }
#pragma unroll
    for (int i = 0; i < LW; i++) {
        const int at = (wave * LW + i) * kWave + lane, r = at / CW, c = at % CW ^ w_swizzle(r);
        int col = min(n0 + 4 * c, width - 4);
        if constexpr (SWIGLU) {  // a wavefront's columns: half of them gates, then the same columns' up projections
            const int of_wave = c / (TN / 4), in_wave = c % (TN / 4), half = in_wave / (TN / 8);
            col = min(n0 + of_wave * (TN / 2) + 4 * (in_wave % (TN / 8)), width - 4) + half * width;
        }
        w_off[i] = ((uint32_t)r * (uint32_t)n + (uint32_t)col) * 4u;
    }
    const char* a_next = reinterpret_cast<const char*>(a + (size_t)m0 * (size_t)k + (size_t)first * kTiledStepF32);
    const char* w_next = reinterpret_cast<const char*>(w + (size_t)first * kTiledStepF32 * (size_t)n);
    const size_t w_step = (size_t)kTiledStepF32 * (size_t)n * 4u;
    const auto load = [&](auto i_, uint32_t stage_at) __attribute__((always_inline)) {  // load i of LOADS
        constexpr int i = decltype(i_)::value;
        if constexpr (i < LA) load_to_lds(stage_at + (wave * LA + i) * 1024, a_next, a_off[i]);
        else load_to_lds(stage_at + kABytes + (wave * LW + i - LA) * 1024, w_next, w_off[i - LA]);
    };
    const auto advance = [&]() __attribute__((always_inline)) {
        a_next += kTiledStepF32 * 4;
        w_next += w_step;
    };

    // Where a lane reads: rows j of A's blocks, chunk 4 sub + g; of W row 4 g + e, columns NI j ... of the wavefront's.
    uint32_t a_at[SUB], w_at[4];
#pragma unroll
    for (int s = 0; s < SUB; s++) a_at[s] = lds0 + (wm * TM + j) * (kTiledStepF32 * 4) + 16 * ((4 * s + g) ^ j / 2 % 8);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int r = 4 * g + e, col = wn * TN + NI * j;
        w_at[e] = lds0 + kABytes + r * (BN * 4) + 16 * (col / 4 ^ w_swizzle(r)) + 4 * (col % 4);
    }

    float4v acc[SUB][MI][NI];  // each half of a step has its own sums
#pragma unroll
    for (int x = 0; x < MI; x++)
#pragma unroll
        for (int y = 0; y < NI; y++) acc[0][x][y] = acc[1][x][y] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    float4v a_reg[2][MI];
    float w_reg[2][4][NI];
    constexpr int READS = MI + 4, PRODUCTS = 4 * MI * NI;
    // read i of READS: the first row of W, the rows of A, the other rows of W -- the order in which the products want them
    const auto read = [&](auto set_, auto sub_, auto i_) __attribute__((always_inline)) {
        constexpr int set = decltype(set_)::value, sub = decltype(sub_)::value, i = decltype(i_)::value;
        if constexpr (i >= 1 && i < 1 + MI) {
            typedef __attribute__((address_space(3))) const float4v* row_ptr;
            a_reg[set][i - 1] = *(row_ptr)(uintptr_t)(a_at[sub] + (i - 1) * 16 * kTiledStepF32 * 4);
        } else {
            constexpr int e = i < 1 ? 0 : i - MI;
            typedef float cols __attribute__((ext_vector_type(NI)));
            typedef __attribute__((address_space(3))) const cols* cols_ptr;
            const cols v = *(cols_ptr)(uintptr_t)(w_at[e] + 16 * sub * BN * 4);
#pragma unroll
            for (int y = 0; y < NI; y++) {
                if constexpr (NI == 1) w_reg[set][e][y] = v.x;
                else w_reg[set][e][y] = v[y];
            }
        }
    };
    // the products of one set of operands; behind them the reads of the other set, over the first three quarters of them, and the loads
    const auto products = [&](auto set_, auto next_sub_, auto load_, uint32_t load_at) __attribute__((always_inline)) {
        constexpr int set = decltype(set_)::value, read_span = PRODUCTS * 3 / 4;
        static_for<PRODUCTS>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value, e = i / (MI * NI), x = i % MI, y = i / MI % NI;
            acc[set][x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(a_reg[set][x][e], w_reg[set][e][y], acc[set][x][y], 0, 0, 0);
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
        const int k0 = (steps - 1) * kTiledStepF32;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int at = (wave * LA + i) * kWave + lane, r = at / CA, c = at % CA ^ r / 2 % 8, past = max(0, k0 + 4 * c - (k - 4));
            load_to_lds(lds0 + (wave * LA + i) * 1024, a + (size_t)m0 * (size_t)k + k0, a_off[i] - 4u * past);
        }
#pragma unroll
        for (int i = 0; i < LW; i++) {
            const int at = (wave * LW + i) * kWave + lane, r = at / CW, past = max(0, k0 + r - (k - 1));
            load_to_lds(lds0 + kABytes + (wave * LW + i) * 1024, w + (size_t)k0 * (size_t)n, w_off[i] - 4u * past * (uint32_t)n);
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
        const int k0 = (steps - 1) * kTiledStepF32;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int at = (wave * LA + i) * kWave + lane, r = at / CA, c = at % CA ^ r / 2 % 8;
            if (k0 + 4 * c >= k) lds_clear16(lds0 + at * 16);
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
        for (int e = 0; e < 4; e++) w_at[e] += by;
        products(one, zero, load_, freed);  // behind the last step it reads what lies in the next buffer, for nobody
    };
    int t = 0;
#pragma unroll 1
    for (; t + STAGES < count; t++) step(true, std::true_type{});
#pragma unroll 1
    for (; t < count; t++) step(t + STAGES == count, std::false_type{});

    // ---- lane (j, g) holds rows 4 g ... 4 g + 3 of every block and its NI neighbouring columns
    typedef float cols __attribute__((ext_vector_type(NI)));
    if constexpr (SWIGLU) {  // lane j has eight lanes' gates, lane j ^ 8 the up projections: each computes two of the four rows
        static_assert(NI >= 2, "sixteen columns would hold no whole chunk of both");
        const bool gates = j < 8;
        const int col = n0 + wn * (TN / 2) + NI * (j % 8);
#pragma unroll
        for (int x = 0; x < MI; x++) {
            float own[4][NI], other[4][NI];
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int y = 0; y < NI; y++) {
                    own[r][y] = acc[0][x][y][r] + acc[1][x][y][r];
                    other[r][y] = dpp_mov<0x128>(own[r][y]);  // row_ror:8
                }
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int row = m0 + wm * TM + 16 * x + 4 * g + (gates ? r : r + 2);
                cols v;
#pragma unroll
                for (int y = 0; y < NI; y++) {
                    const float gate = gates ? own[r][y] : other[r + 2][y], up = gates ? other[r][y] : own[r + 2][y];
                    v[y] = silu_for<float>(gate) * up;
                }
                if (row < m && col < width) *reinterpret_cast<cols*>(out + (size_t)row * (size_t)width + col) = v;
            }
        }
        return;
    }
    float* mine = out + (size_t)blockIdx.y * (size_t)m * (size_t)n;
    const int col = n0 + wn * TN + NI * j;
    if (col >= n) return;  // n is a multiple of 4: NI columns exist together
#pragma unroll
    for (int x = 0; x < MI; x++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = m0 + wm * TM + 16 * x + 4 * g + r;
            if (row >= m) continue;
            cols v;
#pragma unroll
            for (int y = 0; y < NI; y++) {
                if constexpr (NI == 1) v.x = acc[0][x][y][r] + acc[1][x][y][r];
                else v[y] = acc[0][x][y][r] + acc[1][x][y][r];
            }
            *reinterpret_cast<cols*>(mine + (size_t)row * (size_t)n + col) = v;
        }
}

}  // namespace isp
