// What the tiled products for many rows on packed weights share (gemm_tiles_bf16.hip, gemm_tiles_short_bf16.hip): types, and
// which block takes which tile.
#pragma once
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

#define SB() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ uint32_t tiles_pack_bf16(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Which tile block j of XCD x takes, of `rows` token tiles x `cols` columns (a part of k and a row tile; the parts outermost):
// tiles are counted in bands of eight token tiles, a column of the band before the next, and every XCD takes a run of them, as
// long as the others' to one tile.  The 32 blocks that run on an XCD so are about 8 x 4 tiles of one part of k: they share
// their weights and their activations in its L2, and no XCD is left with a round of blocks more than the others.  (With
// whole columns dealt to the XCDs in turn 11 x 20 tiles took two rounds on four of them: 708 us for 2,600 x 5,120 x 17,408,
// 415 now; 5,003 x 5,120 x 17,408 847 -> 800, 5,003 x 34,816 x 5,120 with SwiGLU 1,505 -> 1,478, 2,048 x 28,672 x 4,096 410 -> 407.)
__device__ __forceinline__ bool tiles_place(int tiles, int rows, int cols, int xcd, int j, int& row, int& col) {
    const int per = tiles >> 3, more = tiles & 7;
    if (j >= per + (xcd < more)) return false;
    const int id = xcd * per + min(xcd, more) + j, band = id / (8 * cols), at = id - band * 8 * cols, high = min(8, rows - 8 * band);
    col = at / high;
    row = 8 * band + at % high;
    return true;
}
