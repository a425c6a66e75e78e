// gemm_tile.h -- the f16 planes of activation rows that gemm_tile.hip
// multiplies: device code that writes them, and the buffer's layout.
#pragma once
#include "lkhip_common.h"

// The power of two that brings a row's largest |x| (mx) into [2^14, 2^15)
// (inv) and the one that undoes it (sc), as long as both stay finite and normal:
// below 2^-112 a row's largest lies lower, the smallest normal number at 2^0, where
// the planes' grid of 2^-24 still holds its 24 bits.  A row of zeros takes 2^15.
__device__ __forceinline__ void lk_row_scale(float mx, float& inv, float& sc) {
    int ex = 0;
    (void)frexpf(mx, &ex);  // mx = f * 2^ex, f in [0.5, 1)
    ex = mx == 0.f ? 0 : (ex < -111 ? -111 : (ex > 128 ? 128 : ex));
    inv = ldexpf(1.0f, 15 - ex);
    sc = ldexpf(1.0f, ex - 15);
}

// What 8 scaled values of a lane add to their row's score (the same in every lane of
// the wave; all of them call it).  hi + lo is off by at most max(2^-24 of the value, 2^-25), so
// values below 2^-3 keep fewer than 22 bits.  A row where more than seven eighths
// of the values that are not zero are that small, 2^17 and more below its largest
// (score > 0), is marked, as is one with an infinity, whose lo would be inf - inf:
// gemm_tile_kernel multiplies marked rows with f32 operands.  In a row short of that
// the small values' errors add up to at most 2^-21 of what the others do (root sum of
// squares: sqrt(7) 2^-25.8 against 2^-3), also where the largest meet zero weights;
// f32 operands are off by 2^-20 themselves (8e-7, Q6_K 5632 x 2048).  Fewer would not do:
// SwiGLU rows with gates of 9 and more hold an eighth to a half of such values, which
// add nothing, and took f32 operands at a third of the speed (Q6_K 4096 x 11008, 130
// rows: 545 us).
__device__ __forceinline__ int lk_row_score(const float* v) {
    int s = 0;
#pragma unroll
    for (int e = 0; e < 8; e++)
        s += 8 * __builtin_popcountll(__ballot(v[e] != 0.f && fabsf(v[e]) < 0.125f)) -
             7 * __builtin_popcountll(__ballot(v[e] != 0.f));
    return s;
}
__device__ __forceinline__ bool lk_row_marked(float mx, int score) { return score > 0 || mx == INFINITY; }

// Stores 8 scaled values of row rr of row tile rt, columns 8g .. 8g+7, as f16
// hi + lo where the MFMA operand lane that multiplies them reads them.
__device__ __forceinline__ void lk_store_planes(void* xp, uint32_t rt, uint32_t rr, uint32_t nck, uint32_t g,
                                                const float* v) {
    typedef _Float16 lk_p8 __attribute__((ext_vector_type(8)));
    lk_p8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = (_Float16)v[e];
        lo[e] = (_Float16)(v[e] - (float)hi[e]);
    }
    const uint32_t p = g & 3, j = (p >> 1) | ((p & 1) << 1);  // columns 8p of the block sit in lanes j
    lk_p8* o = (lk_p8*)xp + (((size_t)rt * nck * 4 + (g >> 2)) * 2) * 64 + j * 16 + rr;
    o[0] = hi;
    o[64] = lo;
}
