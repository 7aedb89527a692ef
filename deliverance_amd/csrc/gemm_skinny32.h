// Products of up to 64 rows, 32 columns a workgroup: a kernel of gemm_mfma.hip and, with k shared out over workgroups, of gemm_shares.hip.
#pragma once
#include "gemm_common.h"
#include <da_read_arg.h>

#define SK_LD (64 + 8)       // padded row of a step in LDS, elements (144 bytes)

// ---------------------------------------------------------------------------------------------
// M <= 64 where 16 columns a workgroup would give more workgroups than the chip has compute units (sk_one_a_unit: which
// sizes).  A compute unit pulls in 70 GB/s at best, whatever the pattern, so the bytes of the busiest
// one are what a product of few rows takes: with two workgroups of all rows and 16 columns it pulls the rows of a
// twice.  Here a workgroup owns all rows (row tiles) and `cols` columns, 32 at most, chosen so that every
// compute unit has one; the rest is as above, except that P steps are in flight in registers at any time: a step's
// registers take the step P further on as soon as they are parked.  The same sums in the same order as gemm_skinny with 8
// wavefronts.
// Measured on MI355X with cold weights, K = 1,600, N = 4,800 / 6,400 (16 columns -> 19 / 25): 16 rows 7.1 / 6.8 -> 6.4 / 6.8 us,
// 32 rows 10.0 / 10.4 -> 7.8 / 8.4, 48 rows 11.3 / 13.6 -> 8.6 / 9.3, 64 rows 12.4 / 14.6 -> 10.3 / 10.8.
// ---------------------------------------------------------------------------------------------
// What one lane of a wavefront leaves in LDS another lane of it reads: LDS serves a wavefront's instructions in order, so
// it is the compiler alone that must keep them.
__device__ __forceinline__ void sk_wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// (the vector type of the language: arrays of HIP's uint4, a class, that are only copied stay in memory)
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
// a step's operands, k in elements (a lane past K reads its rows' first piece)
template <int AL, int WL>
__device__ __forceinline__ void sk_fetch(u32x4_t (&av)[AL], u32x4_t (&wv)[WL], const char* a0, const char* w0, const uint32_t (&oa)[AL],
                                         const uint32_t (&ow)[WL], int k, int K) {
  const uint32_t ko = k < K ? 2u * (uint32_t)k : 0u;
#pragma unroll
  for (int u = 0; u < AL; ++u) av[u] = *(const u32x4_t*)(a0 + (oa[u] + ko));
#pragma unroll
  for (int u = 0; u < WL; ++u) wv[u] = *(const u32x4_t*)(w0 + (ow[u] + ko));
}
// ... into the wavefront's piece of LDS, zeros where the lane lies past K
template <int AR, int AL, int WL>
__device__ __forceinline__ void sk_park(const u32x4_t (&av)[AL], const u32x4_t (&wv)[WL], bf16_t* mine, int lr, int lc, bool past) {
#pragma unroll
  for (int u = 0; u < AL; ++u) *(u32x4_t*)&mine[(u * 8 + lr) * SK_LD + lc] = av[u];
#pragma unroll
  for (int u = 0; u < WL; ++u) *(u32x4_t*)&mine[(AR + u * 8 + lr) * SK_LD + lc] = wv[u];
  if (past) {
    const u32x4_t zero = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < AL; ++u) *(u32x4_t*)&mine[(u * 8 + lr) * SK_LD + lc] = zero;
#pragma unroll
    for (int u = 0; u < WL; ++u) *(u32x4_t*)&mine[(AR + u * 8 + lr) * SK_LD + lc] = zero;
  }
}
// AL: loads of 8 rows that cover the workgroup's rows of a (1: up to 8 rows; else two a row tile).
// SHARES: k is shared out over blockIdx.y (gemm_take_share).
template <int AL, int NW, int P, bool SHARES>
__global__ void __launch_bounds__(NW * 64)
gemm_skinny32_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, void* out, int lda, int ldw, int ldo, int M, int N, int K,
                     int cols, int k_share, const void* bias, EpilogueRest er, KvScatter kv) {
  Epilogue ep{bias, er.bias_dtype, er.act, er.accumulate, out, er.out_dtype, ldo};
  if constexpr (SHARES) gemm_take_share(a, w, ep, M, K, k_share);
  constexpr int COLS = 32, MT = (AL + 1) / 2, WL = COLS / 8;    // row tiles of 16; loads of 8 rows that cover w's columns
  constexpr int CT = (COLS + 15) / 16;               // column tiles of 16
  constexpr int AR = MT * 16, TR = AR + COLS;        // rows of a; rows of a step: a's, then w's
  // the wavefronts' partial sums take the place of the parked steps once all products are done
  constexpr int STAGE_BYTES = NW * TR * SK_LD * 2, RED_BYTES = NW * AR * (COLS + 1) * 4;
  __shared__ __attribute__((aligned(16))) char smem[STAGE_BYTES > RED_BYTES ? STAGE_BYTES : RED_BYTES];
  bf16_t (*stage)[TR * SK_LD] = (bf16_t (*)[TR * SK_LD])smem;
  float (*red)[AR][COLS + 1] = (float (*)[AR][COLS + 1])smem;
  const int t = threadIdx.x, lane = t % 64, wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int n0 = blockIdx.x * cols;
  const int n_end = n0 + cols < N ? n0 + cols : N;   // behind the workgroup's last column
  const int lr = lane / 8, lc = (lane % 8) * 8;      // a load: row lr of 8, 16-byte piece lane % 8
  const int fr = lane % 16, fk = (lane / 16) * 8;    // a fragment: row fr of 16, k-group lane / 16
  // byte offsets of the lane's rows behind the first row of a and the workgroup's first of w (64 rows at most: 32 bits hold them)
  const char* const a0 = (const char*)a;
  const char* const w0 = (const char*)(w + (size_t)n0 * ldw);
  uint32_t oa[AL], ow[WL];
#pragma unroll
  for (int i = 0; i < AL; ++i) oa[i] = 2u * (uint32_t)((i * 8 + lr < M ? i * 8 + lr : 0) * lda);
#pragma unroll
  for (int i = 0; i < WL; ++i) ow[i] = 2u * (uint32_t)((n0 + i * 8 + lr < n_end ? i * 8 + lr : 0) * ldw);
  // what the epilogue needs is asked for behind the first steps' operands (its arguments are still on the way when those are asked for),
  // as raw bits from places that always exist
  constexpr int EPT = (AR * COLS + NW * 64 - 1) / (NW * 64);
  uint32_t e_braw[EPT];
  float e_old[EPT];
  int e_slot[EPT];
  const bool bias_bf16 = ep.bias_dtype == DA_BF16;
  floatx4 acc[MT][CT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[i][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16_t* mine = stage[wave];
  // (With AL == 1 the rows 8..15 of the tile are never parked: whatever LDS holds there gives rows of
  // the result that are never stored.)
  // The very last step may be the one that K cuts: lanes past K read the row's first piece instead and park zeros.
  const int steps = (K + 63) / 64;
  const int count = wave < steps ? (steps - wave + NW - 1) / NW : 0;
  u32x4_t av0[AL], wv0[WL], av1[AL], wv1[WL], av2[AL], wv2[WL], av3[AL], wv3[WL];
  const bool cut = K % 64 != 0;
#define SK_FETCH(j, i) sk_fetch(av##j, wv##j, a0, w0, oa, ow, (wave + (i) * NW) * 64 + lc, K);
#define SK_PARK(j, i) sk_park<AR>(av##j, wv##j, mine, lr, lc, cut && (wave + (i) * NW) * 64 + lc >= K);
  auto products = [&]() {
    sk_wave_order();
#pragma unroll
    for (int c = 0; c < 64; c += 32) {
      bf16x8_t wf[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        wf[ct] = __builtin_bit_cast(bf16x8_t, *(const uint4*)&mine[(AR + ct * 16 + fr) * SK_LD + c + fk]);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16x8_t af = __builtin_bit_cast(bf16x8_t, *(const uint4*)&mine[(i * 16 + fr) * SK_LD + c + fk]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[i][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf[ct], acc[i][ct], 0, 0, 0);
      }
    }
    sk_wave_order();
  };
#define SK_EACH(DO)                                     \
  {                                                     \
    DO(0)                                               \
    if constexpr (P > 1) DO(1)                          \
    if constexpr (P > 2) DO(2)                          \
    if constexpr (P > 3) DO(3)                          \
  }
#define SK_FIRST(j) if (j < count) SK_FETCH(j, j)
#define SK_STEADY(j) { SK_PARK(j, i + j) SK_FETCH(j, i + j + P) products(); }
#define SK_LAST(j) if (i + j < count) { SK_PARK(j, i + j) if (i + j + P < count) SK_FETCH(j, i + j + P) products(); }
  static_assert(P >= 1 && P <= 4, "steps in flight");
  SK_EACH(SK_FIRST)
  da_read_arg(ep.act);
  da_read_arg(ep.out_dtype);
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = t + j * NW * 64, m = e / COLS, n = n0 + e % COLS;
    const bool ok = e < AR * COLS && m < M && n < n_end;
    const void* bsrc = (ok && ep.bias) ? ep.bias : (const void*)w;
    const int bidx = (ok && ep.bias) ? n : 0;
    e_braw[j] = bias_bf16 ? (uint32_t)((const bf16_t*)bsrc)[bidx] : ((const uint32_t*)bsrc)[bidx];
    e_old[j] = *((ok && ep.accumulate) ? (const float*)ep.out + (size_t)m * ep.ldo + n : (const float*)w);
    e_slot[j] = *((ok && kv.cache) ? kv.slot_map + m : (const int*)w);
  }
  int i = 0;
  for (; i + 2 * P <= count; i += P) SK_EACH(SK_STEADY)
  for (; i < count; i += P) SK_EACH(SK_LAST)
#undef SK_EACH
#undef SK_FETCH
#undef SK_PARK
#undef SK_FIRST
#undef SK_STEADY
#undef SK_LAST
  lds_barrier();
#pragma unroll
  for (int i2 = 0; i2 < MT; ++i2)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][i2 * 16 + 4 * (lane / 16) + r][ct * 16 + fr] = acc[i2][ct][r];
  lds_barrier();
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = t + j * NW * 64, m = e / COLS, c = e % COLS, n = n0 + c;
    if (e < AR * COLS && m < M && n < n_end) {
      float v = red[0][m][c];
#pragma unroll
      for (int v2 = 1; v2 < NW; ++v2) v += red[v2][m][c];
      const float e_bias = !ep.bias ? 0.f : (bias_bf16 ? __uint_as_float(e_braw[j] << 16) : __uint_as_float(e_braw[j]));
      v = ep.out_dtype == DA_BF16 ? apply_act_bf16(v + e_bias, ep.act) : apply_act(v + e_bias, ep.act);
      const size_t o = (size_t)m * ep.ldo + n;
      if (ep.accumulate) ((float*)ep.out)[o] = e_old[j] + v;
      else if (ep.out_dtype == DA_BF16) ((bf16_t*)ep.out)[o] = f32_to_bf16(v);
      else ((float*)ep.out)[o] = v;
      if (kv.cache && n >= kv.q_cols) kv_column_store(kv, kv_column(kv, n), e_slot[j], v);
    }
  }
}
