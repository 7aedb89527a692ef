// What the norms over rows of the residual stream share (rowwise.hip, norm_rms.hip): how many wavefronts a row takes, and the
// order of its sums.
#pragma once
#include "common.h"

// A row's sum, in every lane.  The row is cut into pieces of 256 columns (a float4 a lane); piece j belongs to partial sum
// j % 4, and the partial sums, each added over its lanes, are added as (0 + 1) + (2 + 3).  With W = 4 wavefronts a row each
// holds one partial sum (its pieces are part[0], part[1], ...; `red` takes the four and is used once), with W = 1 the
// wavefront holds a piece, and so a partial sum, in each entry of `part`: the same bits.
// (The lanes of the four added across the wavefronts first would leave one sum over lanes to W = 1, 5 to 10 % of its
// time with 4,096 rows and more, but a step of few rows waits longer for W = 4: 355M sizes, 33 requests 1,241 -> 1,253 us.)
template <int W, int VPL>
__device__ __forceinline__ float norm_row_sum(const float (&part)[VPL], float* red) {
  static_assert(W == 4 || (W == 1 && VPL <= 4), "a wavefront holds one row's four partial sums at most");
  if (W == 4) {
    float v = part[0];
#pragma unroll
    for (int i = 1; i < VPL; ++i) v += part[i];
    v = wave_sum(v);
    if (threadIdx.x % DA_WAVE == 0) red[threadIdx.x / DA_WAVE] = v;
    lds_barrier();
    return (red[0] + red[1]) + (red[2] + red[3]);
  }
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < VPL; ++i) s[i] = wave_sum(part[i]);
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// What the compiler may fuse or not, written out, so that both ways round alike: the sum of four squares, and a * b + c.
__device__ __forceinline__ float norm_squares(const float4& v) {
#pragma clang fp contract(off)
  return fmaf(v.x, v.x, v.y * v.y) + fmaf(v.z, v.z, v.w * v.w);
}
__device__ __forceinline__ float norm_scaled(float v, float inv, float gain, float add) {
#pragma clang fp contract(off)
  return fmaf(v * inv, gain, add);
}

struct NormGrid {
  int waves, blocks, threads;      // wavefronts a row; the launch
};
// Few rows: four wavefronts a row, the shorter chain of instructions.  Many rows: one, four rows a workgroup; a workgroup a
// row then costs more to start than the row takes, most of all where half or more of its wavefronts have no column.  Up to
// 256 columns one wavefront always.  Else one from `from512` rows on (up to 512 columns), from `from1024` on (up to 1,024).
// us, four wavefronts / one, rows in the caches:
//   256 columns: 64 rows 2.06 / 1.95 (LayerNorm), 2.41 / 2.23 (rms, add, rms); 8,192 rows 6.29 / 3.61, 4.96 / 3.28 (rms), 8.77 / 5.62
//   512: 512 rows 2.28 / 2.34, 768 2.53 / 2.36, 8,192 7.66 / 5.25; rms 1,536 2.51 / 2.57, 2,048 2.69 / 2.69, 8,192 5.85 / 4.64;
//        with the addition 1,536 3.76 / 3.77, 2,048 4.15 / 4.06, 8,192 12.1 / 9.2
//   768: 64 rows 2.06 / 2.30, 768 2.58 / 2.58, 1,024 2.78 / 2.59, 8,192 8.97 / 7.45; rms 2,048 2.99 / 3.20, 4,096 4.50 / 4.39,
//        8,192 7.53 / 7.50 (one wavefront with one sum over lanes: 3.98 and 6.78); with the addition 2,048 4.88 / 5.30, 8,192 14.9 / 17.7
static inline NormGrid norm_grid(int R, int E, int from512, int from1024) {
  const bool one = E <= 256 || R >= (E <= 512 ? from512 : from1024);
  if (!one || E > 1024) return NormGrid{4, R, 4 * DA_WAVE};
  const int rows = R >= 512 ? 4 : 1;
  return NormGrid{1, da_ceil_div(R, rows), rows * DA_WAVE};
}
