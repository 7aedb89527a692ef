// Row-wise kernels: embedding (+ learned positions), LayerNorm (optionally on gathered
// rows), and the write of new keys and values into the paged cache.
#include "norm_common.h"
#include <stdarg.h>

static thread_local char g_error[512] = "";

extern "C" const char* da_last_error() { return g_error; }

void da_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

// ------------------------------------------------------------------------------------------
// x[n, :] = wte[token[n], :] * scale + wpe[pos[n], :]      (32-bit sum, 32-bit result)
// Reference: core/src/main/java/io/teknek/deliverance/model/gpt2/Gpt2Model.java:42-48
// (GPT-2: scale 1; the factor is there for architectures that multiply their embeddings).
// ------------------------------------------------------------------------------------------
__global__ void embed_kernel(const int* __restrict__ tokens, const int* __restrict__ positions,
                             const void* __restrict__ wte, int wte_dtype,
                             const void* __restrict__ wpe, int wpe_dtype,
                             float* __restrict__ x, int E, float scale) {
  const int n = blockIdx.x;
  const size_t trow = (size_t)tokens[n] * E;
  const size_t prow = wpe ? (size_t)positions[n] * E : 0;
  for (int i = threadIdx.x; i < E; i += blockDim.x) {
    float v = load_param(wte, wte_dtype, trow + i);
    if (scale != 1.0f) v *= scale;
    if (wpe) v += load_param(wpe, wpe_dtype, prow + i);
    x[(size_t)n * E + i] = v;
  }
}

extern "C" int da_embed(const int* tokens, const int* positions, const void* wte, int wte_dtype,
                        const void* wpe, int wpe_dtype, float* x, int N, int E, float scale, void* stream) {
  DA_REQUIRE(N >= 0 && E > 0, "embed: bad sizes N=%d E=%d", N, E);
  if (N == 0) return 0;
  int threads = E >= 256 ? 256 : (E >= 128 ? 128 : 64);
  hipLaunchKernelGGL(embed_kernel, dim3(N), dim3(threads), 0, (hipStream_t)stream, tokens, positions,
                     wte, wte_dtype, wpe, wpe_dtype, x, E, scale);
  DA_CHECK_LAUNCH("embed");
  return 0;
}

// ------------------------------------------------------------------------------------------
// dst[r, :] (+)= scale * src[rows ? rows[r] : r, :]: rows gathered, converted between 32-bit and
// bfloat16, or added into the 32-bit residual stream.  For blocks without a norm in front of a
// part, models without a final norm, norms that follow a part, and a part's output that joins the
// stream times a constant (TransformerBlock.java:260-272).
// ------------------------------------------------------------------------------------------
__global__ void copy_rows_kernel(const void* __restrict__ src, int src_dtype, const int* __restrict__ rows,
                                 void* __restrict__ dst, int dst_dtype, int E, int accumulate, float scale) {
  const int r = blockIdx.x;
  const size_t srow = (size_t)(rows ? rows[r] : r) * E, drow = (size_t)r * E;
  for (int i = threadIdx.x; i < E; i += blockDim.x) {
    const float v = load_param(src, src_dtype, srow + i) * scale;
    if (accumulate) ((float*)dst)[drow + i] += v;
    else store_out(dst, dst_dtype, drow + i, v);
  }
}

extern "C" int da_copy_rows(const void* src, int src_dtype, const int* rows, void* dst, int dst_dtype, int R,
                            int E, int accumulate, float scale, void* stream) {
  DA_REQUIRE(R >= 0 && E > 0, "copy_rows: bad sizes R=%d E=%d", R, E);
  DA_REQUIRE(!accumulate || dst_dtype == DA_F32, "copy_rows: accumulation needs a 32-bit destination");
  if (R == 0) return 0;
  const int threads = E >= 256 ? 256 : (E >= 128 ? 128 : 64);
  hipLaunchKernelGGL(copy_rows_kernel, dim3(R), dim3(threads), 0, (hipStream_t)stream, src, src_dtype, rows, dst,
                     dst_dtype, E, accumulate, scale);
  DA_CHECK_LAUNCH("copy_rows");
  return 0;
}

// ------------------------------------------------------------------------------------------
// tokens[n] = sampled[src[n]] where src[n] >= 0: a step that is launched before the step before
// it has been read takes those tokens from that step's sampled tokens on the device.
// ------------------------------------------------------------------------------------------
__global__ void take_tokens_kernel(int* __restrict__ tokens, const int* __restrict__ src,
                                   const int* __restrict__ sampled, int N, int n_sampled, int vocab) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int s = src[n];
  if (s < 0 || s >= n_sampled) return;
  int t = sampled[s];
  t = t < 0 ? 0 : (t >= vocab ? vocab - 1 : t);       // a row that sampled nothing must not index outside the table
  tokens[n] = t;
}

extern "C" int da_take_tokens(int* tokens, const int* src, const int* sampled, int N, int n_sampled, int vocab,
                              void* stream) {
  DA_REQUIRE(N >= 0 && n_sampled > 0 && vocab > 0, "take_tokens: bad sizes N=%d sampled=%d", N, n_sampled);
  if (N == 0) return 0;
  hipLaunchKernelGGL(take_tokens_kernel, dim3(da_ceil_div(N, 64)), dim3(64), 0, (hipStream_t)stream, tokens, src,
                     sampled, N, n_sampled, vocab);
  DA_CHECK_LAUNCH("take_tokens");
  return 0;
}

// ------------------------------------------------------------------------------------------
// Zeros over a buffer of whole 4-byte words (a kernel, so that a recorded step holds no memset node).
// ------------------------------------------------------------------------------------------
__global__ void fill_zero_kernel(uint32_t* __restrict__ p, long n_words) {
  const long stride = (long)gridDim.x * blockDim.x;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n_words; i += stride) p[i] = 0u;
}

extern "C" int da_fill_zero(void* p, long n_bytes, void* stream) {
  DA_REQUIRE(n_bytes >= 0 && n_bytes % 4 == 0 && (uintptr_t)p % 4 == 0, "fill_zero: %ld bytes are not whole words", n_bytes);
  if (n_bytes == 0) return 0;
  const long words = n_bytes / 4;
  const int blocks = (int)(words / 256 < 1 ? 1 : (words / 256 > 2048 ? 2048 : words / 256));
  hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (uint32_t*)p, words);
  DA_CHECK_LAUNCH("fill_zero");
  return 0;
}

// ------------------------------------------------------------------------------------------
// Fixed-size state of the step's sequences, as rows of 4-byte words (any dtype).
//   gather:  out[n, :] = state[slot[seq_of_token[n]], :]   (zeros where the sequence has no slot: a padding row)
//   scatter: state[slot[s], :] = rows[q_start[s+1] - 1, :] for every sequence s that has a slot and brings rows
// A mixer with state reads the first before it walks its rows and calls the second with what each row
// leaves behind: the state of a portion's last row is the request's state after the step.
// ------------------------------------------------------------------------------------------
__global__ void state_gather_kernel(const uint32_t* __restrict__ state, const int* __restrict__ slots,
                                    const int* __restrict__ seq_of_token, uint32_t* __restrict__ out,
                                    int n_slots, int words) {
  const int n = blockIdx.x;
  const int slot = slots[seq_of_token[n]];
  const bool has = slot >= 0 && slot < n_slots;
  for (int i = threadIdx.x; i < words; i += blockDim.x)
    out[(size_t)n * words + i] = has ? state[(size_t)slot * words + i] : 0u;
}

__global__ void state_scatter_kernel(uint32_t* __restrict__ state, const int* __restrict__ slots,
                                     const int* __restrict__ q_start, const uint32_t* __restrict__ rows,
                                     int n_slots, int words) {
  const int s = blockIdx.x;
  const int slot = slots[s], first = q_start[s], last = q_start[s + 1] - 1;
  if (slot < 0 || slot >= n_slots || last < first) return;
  for (int i = threadIdx.x; i < words; i += blockDim.x) state[(size_t)slot * words + i] = rows[(size_t)last * words + i];
}

extern "C" int da_state_gather(const void* state, const int* slots, const int* seq_of_token, void* out, int N,
                               int n_slots, int row_bytes, void* stream) {
  DA_REQUIRE(N >= 0 && n_slots > 0 && row_bytes > 0 && row_bytes % 4 == 0, "state_gather: bad sizes (N=%d, %d slots, rows of %d bytes)",
             N, n_slots, row_bytes);
  if (N == 0) return 0;
  hipLaunchKernelGGL(state_gather_kernel, dim3(N), dim3(row_bytes / 4 >= 256 ? 256 : 64), 0, (hipStream_t)stream,
                     (const uint32_t*)state, slots, seq_of_token, (uint32_t*)out, n_slots, row_bytes / 4);
  DA_CHECK_LAUNCH("state_gather");
  return 0;
}

extern "C" int da_state_scatter(void* state, const int* slots, const int* q_start, const void* rows, int S,
                                int n_slots, int row_bytes, void* stream) {
  DA_REQUIRE(S >= 0 && n_slots > 0 && row_bytes > 0 && row_bytes % 4 == 0, "state_scatter: bad sizes (S=%d, %d slots, rows of %d bytes)",
             S, n_slots, row_bytes);
  if (S == 0) return 0;
  hipLaunchKernelGGL(state_scatter_kernel, dim3(S), dim3(row_bytes / 4 >= 256 ? 256 : 64), 0, (hipStream_t)stream,
                     (uint32_t*)state, slots, q_start, (const uint32_t*)rows, n_slots, row_bytes / 4);
  DA_CHECK_LAUNCH("state_scatter");
  return 0;
}

// ------------------------------------------------------------------------------------------
// LayerNorm over rows of 32-bit x; one wave per row; mean and centred variance in 32-bit.
//   y = (x - mean) / sqrt(var + eps) * w + b        (var biased, eps inside the root)
// Reference: core/src/main/java/io/teknek/deliverance/generator/LayerNorm.java:127-150
// `rows` (optional) gathers: output row r is the norm of input row rows[r].
// ------------------------------------------------------------------------------------------
__global__ void layernorm_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                 const void* __restrict__ w, int w_dtype,
                                 const void* __restrict__ b, int b_dtype, float eps,
                                 void* __restrict__ y, int y_dtype, int R, int E) {
  const int wave = threadIdx.x / DA_WAVE, lane = threadIdx.x % DA_WAVE;
  const int r = blockIdx.x * (blockDim.x / DA_WAVE) + wave;
  if (r >= R) return;
  const float* xr = x + (size_t)(rows ? rows[r] : r) * E;
  float s = 0.f;
  for (int i = lane; i < E; i += DA_WAVE) s += xr[i];
  const float mean = wave_sum(s) / (float)E;
  float q = 0.f;
  for (int i = lane; i < E; i += DA_WAVE) {
    float d = xr[i] - mean;
    q += d * d;
  }
  const float inv = 1.0f / sqrtf(wave_sum(q) / (float)E + eps);
  for (int i = lane; i < E; i += DA_WAVE) {
    float v = (xr[i] - mean) * inv * load_param(w, w_dtype, i);
    if (b) v += load_param(b, b_dtype, i);
    store_out(y, y_dtype, (size_t)r * E + i, v);
  }
}

__device__ __forceinline__ float4 load_param4(const void* p, int dtype, int i) {
  if (dtype == DA_BF16) {
    const uint2 u = *(const uint2*)((const bf16_t*)p + i);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
                       __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u));
  }
  return *(const float4*)((const float*)p + i);
}

// The same norm with the whole row held in registers: every load of the row is in flight at
// once, which is what counts when a step has a handful of rows.  E a multiple of 4, E <= 256 * W * VPL.
// W = 4: a workgroup of four wavefronts is one row, a float4 a lane (two above a width of 1,024): with few rows the chain of
// instructions behind the loads, not the bytes, is what the kernel takes (measured in a recorded chain
// behind the kernel that writes x, one wavefront a row -> four: 64 rows of 768 2.4 -> 2.2 us, of 1,024 2.5 -> 2.1,
// of 1,600 3.1 -> 2.5; 2,048 rows of 1,600 9.4 -> 8.9).
// W = 1: a wavefront a row.  Both give the same bits (norm_row_sum); which one is taken: norm_grid.
// Loads come back in the order they were asked for: the row first, then gain and bias, as raw bits
// that are converted where they are used (a conversion right after its load, or a load inside a
// branch, is waited for on the spot).  PBF16: gain and bias are bfloat16 (else 32-bit); YBF16: y is.
// JOIN: sums that a product left share by share (gemm_take_share) join the row first: x + (((p0 + p1) + ...) + add).
struct RowJoin {
  const float* partial;        // [n][stride]: the sums of the stream's rows, share by share
  long stride;
  int n;                       // 2 to 8
  const void* add;             // a bias a column, or null
  int add_dtype;
  float* keep;                 // where the new row goes (the stream), or null
};
// the sums of 4 columns at entry `at`, the bias of column c
__device__ __forceinline__ float4 join_sums(const RowJoin& j, size_t at, int c) {
  float4 p[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    p[s] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (s < j.n) p[s] = *(const float4*)(j.partial + (size_t)s * j.stride + at);      // (the same for all: a scalar branch)
  }
  uint4 raw = make_uint4(0, 0, 0, 0);
  if (j.add) {
    if (j.add_dtype == DA_BF16) {
      const uint2 u = *(const uint2*)((const bf16_t*)j.add + c);
      raw = make_uint4(u.x << 16, u.x & 0xffff0000u, u.y << 16, u.y & 0xffff0000u);
    } else raw = *(const uint4*)((const float*)j.add + c);
  }
  float4 v = p[0];
#pragma unroll
  for (int s = 1; s < 8; ++s) {
    const bool in = s < j.n;
    v.x = in ? v.x + p[s].x : v.x;
    v.y = in ? v.y + p[s].y : v.y;
    v.z = in ? v.z + p[s].z : v.z;
    v.w = in ? v.w + p[s].w : v.w;
  }
  if (j.add) {
    v.x += __uint_as_float(raw.x);
    v.y += __uint_as_float(raw.y);
    v.z += __uint_as_float(raw.z);
    v.w += __uint_as_float(raw.w);
  }
  return v;
}

// The rows that a kernel reads; those that it may also write (JOIN: the stream, which is `keep` as well) go without the promise
// that no other pointer reaches them.
template <bool JOIN> struct RowSource { typedef const float* __restrict__ type; };
template <> struct RowSource<true> { typedef const float* type; };

template <int VPL, int W, bool PBF16, bool YBF16, bool JOIN = false>
__global__ void __launch_bounds__(4 * DA_WAVE)
layernorm_row_kernel(typename RowSource<JOIN>::type x, const int* __restrict__ rows,
                     const void* __restrict__ w, const void* __restrict__ b,
                     void* __restrict__ y, int E, int R, float eps, RowJoin join) {
  __shared__ float red[2][4];
  constexpr int STRIDE = 4 * W * DA_WAVE;
  const int t = threadIdx.x, c0 = (W == 4 ? t : t % DA_WAVE) * 4;
  const int r = W == 4 ? (int)blockIdx.x : (int)(blockIdx.x * (blockDim.x / DA_WAVE)) + t / DA_WAVE;
  if (W == 1 && r >= R) return;
  const float* xr = x + (size_t)(rows ? rows[r] : r) * E;
  // every load of the row, of the gain and of the bias is asked for at once (past the row's end
  // the row's start is read and left out of the sums), before anything is reduced
  float4 v[VPL];
  uint4 graw[VPL], braw[VPL];           // bfloat16: .x and .y hold the four values
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = c0 + i * STRIDE;
    v[i] = *(const float4*)(xr + (c < E ? c : 0));
  }
  float4 sums[VPL];
  if (JOIN) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = c0 + i * STRIDE, cc = c < E ? c : 0;
      sums[i] = join_sums(join, (size_t)(xr - x) + cc, cc);
    }
  }
  const void* bsrc = b ? b : w;         // without a bias the gain is read twice and dropped
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = c0 + i * STRIDE, cc = c < E ? c : 0;
    if (PBF16) {
      const uint2 g2 = *(const uint2*)((const bf16_t*)w + cc), b2 = *(const uint2*)((const bf16_t*)bsrc + cc);
      graw[i] = make_uint4(g2.x, g2.y, 0, 0);
      braw[i] = make_uint4(b2.x, b2.y, 0, 0);
    } else {
      graw[i] = *(const uint4*)((const float*)w + cc);
      braw[i] = *(const uint4*)((const float*)bsrc + cc);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (JOIN) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = c0 + i * STRIDE;
      v[i].x += sums[i].x; v[i].y += sums[i].y; v[i].z += sums[i].z; v[i].w += sums[i].w;
      if (join.keep && c < E) *(float4*)(join.keep + (size_t)(xr - x) + c) = v[i];
    }
  }
  float part[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) part[i] = c0 + i * STRIDE < E ? (v[i].x + v[i].y) + (v[i].z + v[i].w) : 0.f;
  const float mean = norm_row_sum<W>(part, red[0]) / (float)E;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    v[i].x -= mean; v[i].y -= mean; v[i].z -= mean; v[i].w -= mean;
    part[i] = c0 + i * STRIDE < E ? norm_squares(v[i]) : 0.f;
  }
  const float inv = 1.0f / sqrtf(norm_row_sum<W>(part, red[1]) / (float)E + eps);
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = c0 + i * STRIDE;
    if (c >= E) continue;
    float4 g, bb;
    if (PBF16) {
      g = make_float4(__uint_as_float(graw[i].x << 16), __uint_as_float(graw[i].x & 0xffff0000u),
                      __uint_as_float(graw[i].y << 16), __uint_as_float(graw[i].y & 0xffff0000u));
      bb = make_float4(__uint_as_float(braw[i].x << 16), __uint_as_float(braw[i].x & 0xffff0000u),
                       __uint_as_float(braw[i].y << 16), __uint_as_float(braw[i].y & 0xffff0000u));
    } else {
      g = make_float4(__uint_as_float(graw[i].x), __uint_as_float(graw[i].y), __uint_as_float(graw[i].z), __uint_as_float(graw[i].w));
      bb = make_float4(__uint_as_float(braw[i].x), __uint_as_float(braw[i].y), __uint_as_float(braw[i].z), __uint_as_float(braw[i].w));
    }
    if (!b) bb = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 o = make_float4(norm_scaled(v[i].x, inv, g.x, bb.x), norm_scaled(v[i].y, inv, g.y, bb.y),
                                 norm_scaled(v[i].z, inv, g.z, bb.z), norm_scaled(v[i].w, inv, g.w, bb.w));
    if (YBF16) *(uint2*)((bf16_t*)y + (size_t)r * E + c) = make_uint2(pack2_bf16(o.x, o.y), pack2_bf16(o.z, o.w));
    else *(float4*)((float*)y + (size_t)r * E + c) = o;
  }
}

extern "C" int da_layernorm(const float* x, const int* rows, const void* w, int w_dtype,
                            const void* b, int b_dtype, float eps, void* y, int y_dtype, int R,
                            int E, void* stream) {
  DA_REQUIRE(R >= 0 && E > 0, "layernorm: bad sizes R=%d E=%d", R, E);
  DA_REQUIRE(eps > 0.f, "layernorm: eps must be > 0");
  if (R == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const bool aligned = ((uintptr_t)x % 16 == 0) && ((uintptr_t)y % 16 == 0) && ((uintptr_t)w % 16 == 0) &&
                       (!b || (uintptr_t)b % 16 == 0);
  const bool same = (!b || b_dtype == w_dtype) && (w_dtype == DA_BF16 || w_dtype == DA_F32);   // gain and bias alike
  if (E % 4 == 0 && E <= 2048 && aligned && same) {
    const NormGrid g = norm_grid(R, E, 768, 1024);
#define LN_LAUNCH(V, W, P, Y) hipLaunchKernelGGL((layernorm_row_kernel<V, W, P, Y>), dim3(g.blocks), dim3(g.threads), 0, st, x, rows, w, b, y, E, R, eps, RowJoin{})
#define LN_LAUNCH_Y(V, W, P) do { if (y_dtype == DA_BF16) LN_LAUNCH(V, W, P, true); else LN_LAUNCH(V, W, P, false); } while (0)
#define LN_LAUNCH_P(V, W) do { if (w_dtype == DA_BF16) LN_LAUNCH_Y(V, W, true); else LN_LAUNCH_Y(V, W, false); } while (0)
    if (g.waves == 1) {
      if (E <= 256) LN_LAUNCH_P(1, 1);
      else if (E <= 512) LN_LAUNCH_P(2, 1);
      else LN_LAUNCH_P(4, 1);
    } else if (E <= 1024) LN_LAUNCH_P(1, 4);
    else LN_LAUNCH_P(2, 4);
#undef LN_LAUNCH_P
#undef LN_LAUNCH_Y
#undef LN_LAUNCH
  } else {
    const int waves = 4;
    hipLaunchKernelGGL(layernorm_kernel, dim3(da_ceil_div(R, waves)), dim3(waves * DA_WAVE), 0, st, x, rows, w,
                       w_dtype, b, b_dtype, eps, y, y_dtype, R, E);
  }
  DA_CHECK_LAUNCH("layernorm");
  return 0;
}

// x[r] <- x[r] + (sums of the shares + add) and y[r] <- LayerNorm of the new row, or, with `rows`, y[r] <- LayerNorm of the new
// row rows[r] and x stays as it is (the rows may repeat).  partial: [n][stride], row r of the stream at r * E of each.
static bool join_takes(const void* x, const float* partial, long stride, int n, const void* add, int add_dtype, int E) {
  return E % 4 == 0 && E <= 2048 && n >= 2 && n <= 8 && stride % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)partial % 16 == 0 &&
         (!add || ((add_dtype == DA_BF16 || add_dtype == DA_F32) && (uintptr_t)add % 16 == 0));
}
extern "C" int da_layernorm_join(float* x, const int* rows, const float* partial, long stride, int n, const void* add, int add_dtype,
                                 const void* w, int w_dtype, const void* b, int b_dtype, float eps, void* y, int y_dtype, int R, int E,
                                 void* stream) {
  DA_REQUIRE(R >= 0 && E > 0 && eps > 0.f, "layernorm_join: bad sizes R=%d E=%d eps=%g", R, E, eps);
  DA_REQUIRE(join_takes(x, partial, stride, n, add, add_dtype, E), "layernorm_join: %d shares of rows of %d (2 to 8, a multiple of 4 up to 2,048, 16-byte aligned)", n, E);
  DA_REQUIRE((uintptr_t)y % 16 == 0 && (uintptr_t)w % 16 == 0 && (!b || (uintptr_t)b % 16 == 0) && (!b || b_dtype == w_dtype) &&
             (w_dtype == DA_BF16 || w_dtype == DA_F32) && y_dtype == DA_BF16, "layernorm_join: gain and bias of one type, a bfloat16 result, all 16-byte aligned");
  if (R == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  const RowJoin j{partial, stride, n, add, add_dtype, rows ? nullptr : x};
  const NormGrid g = norm_grid(R, E, 768, 1024);
#define LN_LAUNCH(V, W, P) hipLaunchKernelGGL((layernorm_row_kernel<V, W, P, true, true>), dim3(g.blocks), dim3(g.threads), 0, st, x, rows, w, b, y, E, R, eps, j)
#define LN_LAUNCH_P(V, W) do { if (w_dtype == DA_BF16) LN_LAUNCH(V, W, true); else LN_LAUNCH(V, W, false); } while (0)
  if (g.waves == 1) {
    if (E <= 256) LN_LAUNCH_P(1, 1);
    else if (E <= 512) LN_LAUNCH_P(2, 1);
    else LN_LAUNCH_P(4, 1);
  } else if (E <= 1024) LN_LAUNCH_P(1, 4);
  else LN_LAUNCH_P(2, 4);
#undef LN_LAUNCH_P
#undef LN_LAUNCH
  DA_CHECK_LAUNCH("layernorm_join");
  return 0;
}

// The addition alone, where no such norm follows.
__global__ void __launch_bounds__(256) join_rows_kernel(float* __restrict__ x, int R, int E, RowJoin join) {
  const long c4 = E / 4, i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= R * c4) return;
  const size_t at = (size_t)i * 4;
  float4 v = *(const float4*)(x + at);
  const float4 s = join_sums(join, at, (int)(i % c4) * 4);
  v.x += s.x; v.y += s.y; v.z += s.z; v.w += s.w;
  *(float4*)(x + at) = v;
}
extern "C" int da_join_rows(float* x, const float* partial, long stride, int n, const void* add, int add_dtype, int R, int E, void* stream) {
  DA_REQUIRE(R >= 0 && E > 0 && join_takes(x, partial, stride, n, add, add_dtype, E), "join_rows: bad sizes R=%d E=%d, %d shares", R, E, n);
  if (R == 0) return 0;
  const RowJoin j{partial, stride, n, add, add_dtype, x};
  hipLaunchKernelGGL(join_rows_kernel, dim3(da_ceil_div((long)R * (E / 4), 256)), dim3(256), 0, (hipStream_t)stream, x, R, E, j);
  DA_CHECK_LAUNCH("join_rows");
  return 0;
}

// ------------------------------------------------------------------------------------------
// Keys and values of the step's tokens go to their cache rows.
// qkv: [N, ld] rows holding q | k | v; k starts at column k_off, v at v_off, each Hkv*D wide.
// One cache slot (one layer's pages): [n_pages][2][Hkv][page * D], keys row-major, values
// dimension-major (see common.h); slot_map[n] is page_id * page + row, or -1 for a token whose
// keys are not kept.
// Reference: core/src/main/java/io/teknek/deliverance/generator/CausalSelfAttention.java:315-336
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ void kv_write_kernel(const T* __restrict__ qkv, int ld, int k_off, int v_off,
                                T* __restrict__ cache, const int* __restrict__ slot_map, int Hkv,
                                int D, int page) {
  const int n = blockIdx.x;
  const int slot = slot_map[n];
  if (slot < 0) return;
  const int pg = slot / page, row = slot % page;
  const int W = Hkv * D;
  for (int i = threadIdx.x; i < 2 * W; i += blockDim.x) {
    const int kv = i / W, c = i % W, h = c / D, d = c % D;
    const T v = qkv[(size_t)n * ld + (kv ? v_off : k_off) + c];
    if (kv) cache[cache_v_base(pg, h, Hkv, page, D) + (long long)d * page + row] = v;
    else cache[cache_k_row(pg, h, row, Hkv, page, D) + d] = v;
  }
}

// The same for bfloat16 and many tokens: a workgroup takes 16 consecutive tokens.  Keys go over in
// 16-byte pieces.  Where the 16 tokens fill 16 consecutive, aligned rows of one page (a prompt
// portion that starts on such a boundary), a value column's 16 entries are one 32-byte run in the
// dimension-major page and are stored as such; otherwise entry by entry.
#define KVW_ROWS 16
__global__ void __launch_bounds__(256)
kv_write_rows_kernel(const bf16_t* __restrict__ qkv, int ld, int k_off, int v_off, bf16_t* __restrict__ cache,
                     const int* __restrict__ slot_map, int N, int Hkv, int D, int page) {
  __shared__ int slots[KVW_ROWS];
  __shared__ int run;
  const int n0 = blockIdx.x * KVW_ROWS;
  if (threadIdx.x < KVW_ROWS) slots[threadIdx.x] = n0 + threadIdx.x < N ? slot_map[n0 + threadIdx.x] : -1;
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = slots[0] >= 0 && slots[0] % KVW_ROWS == 0;
    for (int i = 1; i < KVW_ROWS; ++i) ok = ok && slots[i] == slots[0] + i;
    run = ok;
  }
  __syncthreads();
  const int W = Hkv * D, chunks = W / 8;
  // blockIdx.y splits the columns, so that few tokens still fill the chip
  const int t = threadIdx.x + blockIdx.y * blockDim.x, stride = blockDim.x * gridDim.y;
  // keys: rows of 16-byte pieces
  for (int e = t; e < KVW_ROWS * chunks; e += stride) {
    const int i = e / chunks, c = (e % chunks) * 8, slot = slots[i];
    if (slot < 0) continue;
    const int h = c / D, d = c % D;
    *(uint4*)(cache + cache_k_row(slot / page, h, slot % page, Hkv, page, D) + d) =
        *(const uint4*)(qkv + (size_t)(n0 + i) * ld + k_off + c);
  }
  // values: a thread takes a column (head, dimension) of the 16 tokens
  for (int c = t; c < W; c += stride) {
    const int h = c / D, d = c % D;
    bf16_t v[KVW_ROWS];
#pragma unroll
    for (int i = 0; i < KVW_ROWS; ++i) v[i] = slots[i] >= 0 ? qkv[(size_t)(n0 + i) * ld + v_off + c] : (bf16_t)0;
    if (run) {
      bf16_t* dst = cache + cache_v_base(slots[0] / page, h, Hkv, page, D) + (long long)d * page + slots[0] % page;
      uint32_t u[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) u[i] = (uint32_t)v[2 * i] | ((uint32_t)v[2 * i + 1] << 16);
      *(uint4*)dst = make_uint4(u[0], u[1], u[2], u[3]);
      *(uint4*)(dst + 8) = make_uint4(u[4], u[5], u[6], u[7]);
    } else {
#pragma unroll
      for (int i = 0; i < KVW_ROWS; ++i)
        if (slots[i] >= 0)
          cache[cache_v_base(slots[i] / page, h, Hkv, page, D) + (long long)d * page + slots[i] % page] = v[i];
    }
  }
}

extern "C" int da_kv_write(const void* qkv, int dtype, int ld, int k_off, int v_off, void* cache,
                           const int* slot_map, int N, int Hkv, int D, int page, void* stream) {
  DA_REQUIRE(N >= 0 && Hkv > 0 && D > 0 && page > 0, "kv_write: bad sizes");
  DA_REQUIRE(k_off >= 0 && v_off >= 0 && k_off + Hkv * D <= ld && v_off + Hkv * D <= ld,
             "kv_write: k/v columns [%d,%d)+%d exceed the row length %d", k_off, v_off, Hkv * D, ld);
  if (N == 0) return 0;
  const int threads = 256;
  const bool vec = dtype == DA_BF16 && N >= 256 && D % 8 == 0 && page % KVW_ROWS == 0 && ld % 8 == 0 &&
                   k_off % 8 == 0 && ((uintptr_t)qkv % 16 == 0) && ((uintptr_t)cache % 16 == 0);
  if (vec)
    hipLaunchKernelGGL(kv_write_rows_kernel, dim3(da_ceil_div(N, KVW_ROWS), da_ceil_div(Hkv * D, 256)), dim3(threads), 0, (hipStream_t)stream,
                       (const bf16_t*)qkv, ld, k_off, v_off, (bf16_t*)cache, slot_map, N, Hkv, D, page);
  else if (dtype == DA_BF16)
    hipLaunchKernelGGL(kv_write_kernel<bf16_t>, dim3(N), dim3(threads), 0, (hipStream_t)stream,
                       (const bf16_t*)qkv, ld, k_off, v_off, (bf16_t*)cache, slot_map, Hkv, D, page);
  else
    hipLaunchKernelGGL(kv_write_kernel<float>, dim3(N), dim3(threads), 0, (hipStream_t)stream,
                       (const float*)qkv, ld, k_off, v_off, (float*)cache, slot_map, Hkv, D, page);
  DA_CHECK_LAUNCH("kv_write");
  return 0;
}
