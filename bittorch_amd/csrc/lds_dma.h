// Loads from global memory straight into LDS, and the remainder rule of the tiled GEMMs built on them.
#pragma once

#include "bt_common.h"

namespace bt {

// The compiler does not see these loads: whoever uses them waits for them (vmcnt) by hand.  M0's 16 bits hold the LDS byte
// offset, so the area they write ends below 64 KiB.
// 16 (4) bytes a lane from sbase + voff to LDS byte lds_off + 16 (4) * lane
__device__ __forceinline__ void dma16(uint32_t lds_off, uint32_t voff, const void* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_off)), "v"(voff), "s"(sbase) : "memory");
}
__device__ __forceinline__ void dma4(uint32_t lds_off, uint32_t voff, const void* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_off)), "v"(voff), "s"(sbase) : "memory");
}

// Where a wave's packed weights come from, per stage of 64 k: 16 rows of 64 columns of row-major W_T, lane (j, g) decoding the
// four bytes of its columns 4 j .. +3 in its rows 4 g .. +3.
//   W_ROWS    four 4-byte loads a lane, a row each; LDS holds [r][lane]
//   W_ROWS16  N % 16 == 0 and W_T 16-byte aligned: one 16-byte load a lane (row rows16_row(lane), columns 16 (lane % 4) .. +15),
//             so that LDS holds the same [r][lane].  A quarter of the requests: 2048 x 4096 x 4096 bf16 59 -> 54 us
//   W_TILES   the decode-tiled copy, W_FIELDS its field layout: one 16-byte load a lane, its four columns
enum { W_ROWS = 0, W_ROWS16 = 1, W_TILES = 2, W_FIELDS = 3 };
__device__ __forceinline__ int rows16_row(int lane) { return 4 * ((lane >> 2) & 3) + (lane >> 4); }  // lane (j, g) / 4 of LDS row r
static inline int w_source(bool tiled, bool fields, const void* W, int64_t N) {
    if (tiled) return fields ? W_FIELDS : W_TILES;
    return N % 16 == 0 && ((uintptr_t)W) % 16 == 0 ? W_ROWS16 : W_ROWS;
}

// Option GEMM_TAIL_SPLIT = 0 (tests, A/B runs): every tile of every launch has 128 rows.
static inline bool gemm_whole_tiles() {
    const char* env = option(OPT_GEMM_TAIL_SPLIT);
    return env && env[0] == '0';
}
// Into how many finer ones the last, incomplete round of an XCD's 128-row tiles is cut (two workgroups per compute unit).
// Two workgroups that end together free their compute unit for the next two, so a remainder of whole tiles runs in pairs on a
// part of the chip.  Measured (int8, row-major weights, us, whole / halves / quarters; remainder of 64): 2048 x 11008 x 4096
// (22) 104 / 97 / 111; 2900 x 6400 x 6400 (8) 136 / 120 / 122, tiled 120 / 112 / 106; 4096 x 4100 x 4096 (4) 98 / 88 / 86;
// 2304 x 4096 x 4096 (36) 56 / 63 / 80.
static inline int gemm_dma_parts(int64_t tiles) {
    if (gemm_whole_tiles()) return 1;
    const int64_t slots = 2 * gemm_compute_units() / 8, rem = ceil_div(tiles, 8) % slots;
    return rem == 0 || 2 * rem > slots ? 1 : 5 * rem > slots ? 2 : 4;
}

}  // namespace bt
