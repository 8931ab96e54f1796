// What the tiled products (linear_tiled.h, linear_tiled_f32.h) and the attention of prompts share: loads from memory straight into LDS,
// reads of matrix operands from there, and loops whose index is a constant.
#pragma once

#include <type_traits>

#include "isp_common.h"

namespace isp {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// 16 bytes per lane from base + off into LDS, lane i's to lds + 16 i.  An asm statement because the compiler would make every later
// LDS read wait for all such loads; the kernel waits by itself (wait_loads).  Nothing is written but LDS: no register is in flight.
// s_nop: M0 must not be written in the instruction right before.
__device__ __forceinline__ void load_to_lds(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(off), "s"(base) : "memory");
}
// until at most N of this wavefront's loads are outstanding (they arrive in order)
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ half4 lds_read_transposed(uint32_t at) {
    typedef short short4v __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4v* lds_ptr;
    const short4v r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(uintptr_t)at);
    return __builtin_bit_cast(half4, r);
}
__device__ __forceinline__ half8 lds_read_row(uint32_t at) {
    typedef __attribute__((address_space(3))) const half8* lds_ptr;
    return *(lds_ptr)(uintptr_t)at;
}
__device__ __forceinline__ void lds_clear16(uint32_t at) {
    typedef __attribute__((address_space(3))) float4v* lds_ptr;
    *(lds_ptr)(uintptr_t)at = float4v{0.0f, 0.0f, 0.0f, 0.0f};
}

// Which tile this workgroup takes.  Workgroups are handed to the eight XCDs in turn; each XCD gets a contiguous run of tiles, four rows of
// tiles at a time, so that its L2 holds what its workgroups share.  (Eight rows of tiles: within 2 % of it either way.)
struct TilePlace {
    int row, col;
};
__device__ __forceinline__ TilePlace place_tile(int rows_of_tiles, int cols_of_tiles) {
    constexpr int kXcds = 8, kTileRows = 4;
    const int tiles = rows_of_tiles * cols_of_tiles, per_xcd = tiles / kXcds, xcd = (int)blockIdx.x % kXcds;
    const int index = xcd * per_xcd + min(xcd, tiles % kXcds) + (int)blockIdx.x / kXcds;
    const int band = index / (kTileRows * cols_of_tiles), in_band = index - band * kTileRows * cols_of_tiles;
    const int band_rows = min(kTileRows, rows_of_tiles - band * kTileRows);
    return {band * kTileRows + in_band % band_rows, in_band / band_rows};
}

}  // namespace isp
