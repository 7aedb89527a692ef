// What the norms over rows of the residual stream share (rowwise.hip, norm_rms.hip): how many wavefronts a row takes, and the
// order of its sums.
#pragma once
#include "common.h"

// A row's sum, in every lane.  The row is cut into pieces of 256 columns (a float4 a lane); piece j belongs to partial sum
// j % 4 of its lane, a lane's partial sums are added as (0 + 1) + (2 + 3), and the lanes follow.  With W = 4 wavefronts a row
// each holds one partial sum (its pieces are part[0], part[1], ...; they meet in `red`, which is used once), with W = 1 a
// lane holds a piece, and so a partial sum, in each entry of `part`: the same bits.
template <int W, int VPL>
__device__ __forceinline__ float norm_row_sum(const float (&part)[VPL], float* red) {
  static_assert(W == 4 || (W == 1 && VPL <= 4), "a lane holds four partial sums at most");
  if (W == 4) {
    const int t = threadIdx.x, lane = t % DA_WAVE;
    float v = part[0];
#pragma unroll
    for (int i = 1; i < VPL; ++i) v += part[i];
    red[t] = v;
    lds_barrier();
    return wave_sum((red[lane] + red[DA_WAVE + lane]) + (red[2 * DA_WAVE + lane] + red[3 * DA_WAVE + lane]));
  }
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < VPL; ++i) s[i] = part[i];
  return wave_sum((s[0] + s[1]) + (s[2] + s[3]));
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
//   256 columns: 64 rows 2.04 / 1.93 (LayerNorm), 2.62 / 2.23 (rms, add, rms); 8,192 rows 5.72 / 3.55, 4.73 / 3.28 (rms), 8.61 / 5.59
//   512: 768 rows 2.28 / 2.32, 1,024 2.40 / 2.37, 8,192 6.90 / 4.81; rms 1,024 2.30 / 2.31, 1,536 2.54 / 2.44, 8,192 5.69 / 4.48;
//        with the addition 1,024 3.30 / 3.42, 1,536 3.91 / 3.81, 8,192 13.4 / 8.9
//   768: 64 rows 2.08 / 2.17, 1,024 2.53 / 2.46, 1,536 3.02 / 2.94, 8,192 8.62 / 6.80 (1,024 columns: 1,024 rows 2.67 / 2.75);
//        rms 2,048 3.01 / 3.08, 4,096 4.42 / 3.97, 8,192 7.53 / 6.75; with the addition 2,048 5.01 / 5.52, 4,096 7.89 / 7.66,
//        8,192 16.0 / 17.9
static inline NormGrid norm_grid(int R, int E, int from512, int from1024) {
  const bool one = E <= 256 || R >= (E <= 512 ? from512 : from1024);
  if (!one || E > 1024) return NormGrid{4, R, 4 * DA_WAVE};
  const int rows = R >= 512 ? 4 : 1;
  return NormGrid{1, da_ceil_div(R, rows), rows * DA_WAVE};
}
