// Root-mean-square norms over rows of the 32-bit residual stream, all in 32-bit:
//
//   rms(x)[i] = x[i] / sqrt(mean(x^2) + eps) * (offset + w[i])
//
// `offset` is 0 for a gain stored as it is applied and 1 for a gain stored around zero.  Four wavefronts or one own a
// row (norm_grid); where the width allows it the whole row sits in registers, so every load is in flight
// at once and the row is read once.
//
//   da_rmsnorm      y = rms(x[rows[r]] or x[r])                       (32-bit or bfloat16 out)
//   da_rmsnorm_add  x += rms_a(src);  h = rms_b(x), or x itself converted (optional)   the norm behind a part, the residual
//                   addition and the norm in front of the next part in one pass over the row
#include "norm_common.h"
#include <limits.h>

// Four entries of a gain as raw bits (bfloat16: .x and .y hold them), converted where they are used: a conversion right
// behind its load would be waited for on the spot.
__device__ __forceinline__ uint4 rms_raw4(const void* p, int dtype, int i) {
  if (dtype == DA_BF16) {
    const uint2 u = *(const uint2*)((const bf16_t*)p + i);
    return make_uint4(u.x, u.y, 0, 0);
  }
  return *(const uint4*)((const float*)p + i);
}
__device__ __forceinline__ float4 rms_gain4(const uint4& u, int dtype) {
  const bool h = dtype == DA_BF16;
  return make_float4(__uint_as_float(h ? u.x << 16 : u.x), __uint_as_float(h ? u.x & 0xffff0000u : u.y),
                     __uint_as_float(h ? u.y << 16 : u.z), __uint_as_float(h ? u.y & 0xffff0000u : u.w));
}

__device__ __forceinline__ void rms_store4(void* y, int y_dtype, size_t at, float4 o) {
  if (y_dtype == DA_BF16) {
    *(uint2*)((bf16_t*)y + at) = make_uint2(pack2_bf16(o.x, o.y), pack2_bf16(o.z, o.w));
  } else {
    *(float4*)((float*)y + at) = o;
  }
}

// VPL float4 a lane: W wavefronts a row (4, or 1): E a multiple of 4, E <= 256 * W * VPL.  ADD: src is normalised with (wa), added into x,
// and (if h) the new x is normalised with (wb) into h.  !ADD: y = rms(x) with wa.
template <int VPL, int W, bool ADD>
__global__ void __launch_bounds__(4 * DA_WAVE)
rmsnorm_row_kernel(const float* __restrict__ src, const int* __restrict__ rows, const void* __restrict__ wa, float* __restrict__ x,
                   const void* __restrict__ wb, void* __restrict__ y, int E, int dtypes, int R, float offset, float eps) {
  // (the first 14 words, with the three types in one, are in registers when the wavefront starts: build.py, KERNARG_PRELOAD)
  const int wa_dtype = dtypes & 0xff, wb_dtype = (dtypes >> 8) & 0xff, y_dtype = dtypes >> 16;
  __shared__ float red[2][4];
  constexpr int STRIDE = 4 * W * DA_WAVE;
  const int t = threadIdx.x, c0 = (W == 4 ? t : t % DA_WAVE) * 4;
  const int r = W == 4 ? (int)blockIdx.x : (int)(blockIdx.x * (blockDim.x / DA_WAVE)) + t / DA_WAVE;
  if (W == 1 && r >= R) return;
  const float* sr = src + (size_t)(rows ? rows[r] : r) * E;
  // the gains are asked for beside the rows, so that the kernel costs one round trip to memory and not one per norm
  float4 v[VPL], xv[VPL];
  uint4 ga[VPL], gb[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = c0 + i * STRIDE;
    v[i] = *(const float4*)(sr + (c < E ? c : 0));
    if (ADD) xv[i] = *(const float4*)(x + (size_t)r * E + (c < E ? c : 0));
  }
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = c0 + i * STRIDE, cc = c < E ? c : 0;
    ga[i] = rms_raw4(wa, wa_dtype, cc);
    if (ADD && y && wb) gb[i] = rms_raw4(wb, wb_dtype, cc);
  }
  __builtin_amdgcn_sched_barrier(0);                   // the loads stay ahead of the sums
  float part[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) part[i] = c0 + i * STRIDE < E ? norm_squares(v[i]) : 0.f;
  const float inv = 1.0f / sqrtf(norm_row_sum<W>(part, red[0]) / (float)E + eps);
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = c0 + i * STRIDE;
    if (c < E) {
      const float4 g = rms_gain4(ga[i], wa_dtype);
      const float4 old = ADD ? xv[i] : make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 o = make_float4(norm_scaled(v[i].x, inv, offset + g.x, old.x), norm_scaled(v[i].y, inv, offset + g.y, old.y),
                                   norm_scaled(v[i].z, inv, offset + g.z, old.z), norm_scaled(v[i].w, inv, offset + g.w, old.w));
      if (ADD) {
        *(float4*)(x + (size_t)r * E + c) = o;
        xv[i] = o;
        part[i] = norm_squares(o);                     // (past the row's end it stays 0)
      } else {
        rms_store4(y, y_dtype, (size_t)r * E + c, o);
      }
    }
  }
  if (ADD && y && !wb) {                               // no second norm: the new x itself, converted
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = c0 + i * STRIDE;
      if (c < E) rms_store4(y, y_dtype, (size_t)r * E + c, xv[i]);
    }
  } else if (ADD && y) {
    const float inv2 = 1.0f / sqrtf(norm_row_sum<W>(part, red[1]) / (float)E + eps);
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = c0 + i * STRIDE;
      if (c < E) {
        const float4 g = rms_gain4(gb[i], wb_dtype);
        rms_store4(y, y_dtype, (size_t)r * E + c,
                   make_float4(xv[i].x * inv2 * (offset + g.x), xv[i].y * inv2 * (offset + g.y),
                               xv[i].z * inv2 * (offset + g.z), xv[i].w * inv2 * (offset + g.w)));
      }
    }
  }
}

// any width, any alignment
template <bool ADD>
__global__ void rmsnorm_any_kernel(const float* __restrict__ src, const int* __restrict__ rows, const void* __restrict__ wa,
                                   int wa_dtype, float* __restrict__ x, const void* __restrict__ wb, int wb_dtype,
                                   float offset, float eps, void* __restrict__ y, int y_dtype, int R, int E) {
  const int lane = threadIdx.x % DA_WAVE;
  const int r = blockIdx.x * (blockDim.x / DA_WAVE) + threadIdx.x / DA_WAVE;
  if (r >= R) return;
  const float* sr = src + (size_t)(rows ? rows[r] : r) * E;
  float q = 0.f;
  for (int i = lane; i < E; i += DA_WAVE) q += sr[i] * sr[i];
  const float inv = 1.0f / sqrtf(wave_sum(q) / (float)E + eps);
  float q2 = 0.f;
  for (int i = lane; i < E; i += DA_WAVE) {
    float o = sr[i] * inv * (offset + load_param(wa, wa_dtype, i));
    if (ADD) {
      o += x[(size_t)r * E + i];
      x[(size_t)r * E + i] = o;
      q2 += o * o;
    } else {
      store_out(y, y_dtype, (size_t)r * E + i, o);
    }
  }
  if (ADD && y && !wb) {
    for (int i = lane; i < E; i += DA_WAVE) store_out(y, y_dtype, (size_t)r * E + i, x[(size_t)r * E + i]);
  } else if (ADD && y) {
    const float inv2 = 1.0f / sqrtf(wave_sum(q2) / (float)E + eps);
    for (int i = lane; i < E; i += DA_WAVE)
      store_out(y, y_dtype, (size_t)r * E + i, x[(size_t)r * E + i] * inv2 * (offset + load_param(wb, wb_dtype, i)));
  }
}

template <bool ADD>
static void rms_launch(const float* src, const int* rows, const void* wa, int wa_dtype, float* x, const void* wb,
                       int wb_dtype, float offset, float eps, void* y, int y_dtype, int R, int E, hipStream_t st) {
  const bool aligned = ((uintptr_t)src % 16 == 0) && ((uintptr_t)y % 16 == 0) && ((uintptr_t)wa % 16 == 0) &&
                       ((uintptr_t)wb % 16 == 0) && ((uintptr_t)x % 16 == 0);
#define RMS_LAUNCH(V, W)                                                                                             \
  hipLaunchKernelGGL((rmsnorm_row_kernel<V, W, ADD>), dim3(g.blocks), dim3(g.threads), 0, st, src, rows, wa, x, wb, y, E, \
                     wa_dtype | wb_dtype << 8 | y_dtype << 16, R, offset, eps)
  if (E % 4 == 0 && E <= 4096 && aligned) {
    const NormGrid g = norm_grid(R, E, 2048, ADD ? INT_MAX : 4096);
    if (g.waves == 1) {
      if (E <= 256) RMS_LAUNCH(1, 1);
      else if (E <= 512) RMS_LAUNCH(2, 1);
      else RMS_LAUNCH(4, 1);
    } else if (E <= 1024) RMS_LAUNCH(1, 4);
    else if (E <= 2048) RMS_LAUNCH(2, 4);
    else RMS_LAUNCH(4, 4);
  } else {
    hipLaunchKernelGGL((rmsnorm_any_kernel<ADD>), dim3(da_ceil_div(R, 4)), dim3(4 * DA_WAVE), 0, st, src, rows, wa,
                       wa_dtype, x, wb, wb_dtype, offset, eps, y, y_dtype, R, E);
  }
#undef RMS_LAUNCH
}

extern "C" int da_rmsnorm(const float* x, const int* rows, const void* w, int w_dtype, float offset, float eps, void* y,
                          int y_dtype, int R, int E, void* stream) {
  DA_REQUIRE(R >= 0 && E > 0, "rmsnorm: bad sizes R=%d E=%d", R, E);
  DA_REQUIRE(eps > 0.f, "rmsnorm: eps must be > 0");
  DA_REQUIRE(x && w && y, "rmsnorm: a null operand");
  if (R == 0) return 0;
  rms_launch<false>(x, rows, w, w_dtype, nullptr, nullptr, 0, offset, eps, y, y_dtype, R, E, (hipStream_t)stream);
  DA_CHECK_LAUNCH("rmsnorm");
  return 0;
}

extern "C" int da_rmsnorm_add(const float* src, const void* wa, int wa_dtype, float* x, const void* wb, int wb_dtype,
                              float offset, float eps, void* h, int h_dtype, int R, int E, void* stream) {
  DA_REQUIRE(R >= 0 && E > 0, "rmsnorm_add: bad sizes R=%d E=%d", R, E);
  DA_REQUIRE(eps > 0.f, "rmsnorm_add: eps must be > 0");
  DA_REQUIRE(src && wa && x && (const float*)x != src, "rmsnorm_add: a null operand, or the part's output is the stream itself");
  DA_REQUIRE(h != nullptr || wb == nullptr, "rmsnorm_add: the second norm needs an output");
  if (R == 0) return 0;
  rms_launch<true>(src, nullptr, wa, wa_dtype, x, wb, wb_dtype, offset, eps, h, h_dtype, R, E, (hipStream_t)stream);
  DA_CHECK_LAUNCH("rmsnorm_add");
  return 0;
}
