// 32-bit matrix products on the gfx950 matrix cores:
//
//   out[m, n] (+)= act( sum_k a[m, k] * w[n, k] + bias[n] )
//
// a [M, K], w [N, K] and out are 32-bit, K contiguous and a multiple of 4; nothing is rounded to fewer bits
// (v_mfma_f32_16x16x4_f32 multiplies and adds in 32-bit).  A q|k|v product also writes its k and v columns to the rows'
// places in the paged cache.
//
// Every output element sums over k in one order, whatever M is and whichever kernel computes it: k goes in chunks of
// 128, a chunk in 8 groups of 16, and a group in 4 instructions of which instruction j takes the k with k % 4 = j (lane
// l of a fragment holds row or column l % 16 and loads the 4 consecutive k from 4 * (l / 16) in one 16-byte piece); the
// sum of a chunk starts from zero and joins the total of the chunks before it.  (Two levels: a long sum into one
// 32-bit accumulator loses about sqrt(K) roundings, this one sqrt(128) + sqrt(K / 128).)
//
//  * gemm_f32_rows: few rows.  A workgroup owns 4, 8 or 16 rows and as many columns as give every compute unit one workgroup (16 at
//    most); its wavefronts take whole chunks, from memory through their own pieces of LDS into fragments, and the chunks' sums are
//    added through LDS.  Bound by the bytes of w.
//  * gemm_f32_ln_rows: the same with a LayerNorm in front (da_gemm_f32_ln).
//  * gemm_f32_rows_direct: few rows, from memory straight into fragments; where that is ahead (f32_rows_staged).
//  * gemm_f32_tile: block tiles of 64 x 64 or 32 x 32 through two LDS buffers, slabs of 32 k, the next four slabs in flight
//    in registers.  Bound by the matrix cores (157 TFLOP/s in 32-bit) where the tiles fill the chip several times over:
//    1,000 x 50,257 x 768 in 687 us, 72 % of that rate; below, by the latency of a slab, which small tiles, several of
//    them on a compute unit, hide better than large ones (526 x 3,072 x 768: 32 x 32 31 us, 64 x 64 34, 128 x 128 72).
//
// Measured on MI355X with cold weights, us, gemm_f32_rows_direct -> gemm_f32_rows: 4 rows, K x N 768 x 768 4.5 -> 3.8, 768 x 2,304 5.3 -> 4.7, 768 x 3,072 5.6 -> 5.2, 3,072 x 768 10.8 -> 6.1,
// 768 x 50,257 39.9 -> 32.1; 8 rows, 3,072 x 768 12.0 -> 7.7; 16 rows 13.8 -> 9.6; 64 rows 14.3 -> 11.4; 32 rows, 768 x 3,072 8.7 -> 7.9.
// Tiles: 526 x 768 x 3,072 38, 526 x 2,304 x 768 27, 526 x 50,257 x 768 392.
#include "gemm_common.h"
#include "norm_common.h"
#include <da_read_arg.h>
#include <type_traits>

#define GF_CHUNK 128
#define GF_BK 32
#define GF_ROWS_CAP 50
#define GF_ROWS_MAX_K (GF_ROWS_CAP * GF_CHUNK)      // the chunks' sums of 16 x 16 outputs fit in 64 KB of LDS
#define GF_LD (GF_BK + 4)    // padded LDS row, floats (144 bytes): 16 consecutive rows start in different banks

__device__ __forceinline__ float4 gf_load(const float* p) { return *(const float4*)p; }

__device__ __forceinline__ floatx4 gf_group(const float4& a, const float4& w, floatx4 c) {      // the 16 k of a group
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, w.x, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, w.y, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, w.z, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, w.w, c, 0, 0, 0);
}
// What one lane of a wavefront leaves in LDS another lane of it reads: LDS serves a wavefront's instructions in order, so
// it is the compiler alone that must keep them.
__device__ __forceinline__ void gf_wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}


// An output element's bias, old value, place in the cache and the column's offset in a page.
#define GF_EPILOGUE_LOADS                                                                                                      \
  da_read_arg(ep.act);                                                                                                         \
  const float e_bias_raw = (e_ok && ep.bias) ? load_param(ep.bias, ep.bias_dtype, en) : 0.f;                                   \
  const float e_old = *((e_ok && ep.accumulate) ? (const float*)ep.out + (size_t)em * ep.ldo + en : w);                        \
  const int e_slot = *((e_ok && kv.cache) ? kv.slot_map + em : (const int*)w);                                                 \
  KvColumn e_col;                                                                                                              \
  if (kv.cache) e_col = kv_column(kv, en);

// ---------------------------------------------------------------------------------------------
// Few rows: blockIdx.x: `cols` columns (4 WL at most), blockIdx.y: 4 AL rows.  A wavefront takes sets of P chunks, v, v + NW,
// ...; a set's loads (2 rows x 512 bytes each, whole cache lines) are in flight while the set before it is multiplied, and pass
// through the wavefront's own piece of LDS into fragments.  A product of 16 x 16 holds P chunks side by side: chunk p has the
// rows and the columns from p * 16 / P on, and what one chunk's rows give with another's columns is dropped.  So 4 rows and 4
// columns take a quarter of the matrix instructions that a chunk at a time would.
// Bound by the bytes of w where the columns are many; else by the chain launch, load, products, sums.
// ---------------------------------------------------------------------------------------------
// The 16-byte piece kk of a parked row: turned by the row's place in the fragment, so that the writes (32 pieces of a row) and
// the reads (one piece of 16 rows) both spread over the banks.
// (the vector type of the language: arrays of HIP's float4, a class, that are only copied stay in memory)
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
__device__ __forceinline__ int gf_place(int row, int kk) { return row * 32 + (kk ^ (row & 15)); }
// CAP: chunks that the partial sums in LDS have room for.
//
// LN: a's rows are normalised first (LayerNorm of the stream's rows, up to GF_LN_MAX_K columns: a set a wavefront at most, so that
// all of a is in registers).  The sums of layernorm_row_kernel's order (norm_common.h): a piece of 256 columns is two chunks, its
// sum over the lanes (l0 + l1) + (l2 + l3) of 16 lanes each, so the product's operands have the bits that the two kernels give.
#define GF_LN_MAX_K 1024
struct GfNorm {
  const float* g;
  const float* b;
  float eps;
};
template <int WL, int AL, int NW, int CAP, bool LN>
__device__ __forceinline__ void
gemm_f32_rows_body(const float* __restrict__ a, const float* __restrict__ w, int lda, int ldw, int M, int N, int K, int n_chunks, int cols,
                   const Epilogue& ep, const KvScatter& kv, const GfNorm& norm) {
  constexpr int P = WL == 1 && AL == 1 ? 4 : (WL <= 2 && AL <= 2 ? 2 : 1), S = 16 / P;    // chunks of a product; rows and columns of each
  constexpr int RA = 4 * AL, CW = 4 * WL, LA = RA / 2, LW = CW / 2;     // rows, columns; loads a chunk
  static_assert(RA <= S && CW <= S, "a chunk's rows and columns fit their part of the fragments");
  static_assert(NW * 64 >= RA * CW, "a thread an output");
  __shared__ __attribute__((aligned(16))) f32x4_t gf_stage[NW][P * (RA + CW) * 32];
  __shared__ float gf_red[CAP * RA * (CW + 1)];                        // [n_chunks][RA][CW + 1]
  const int t = threadIdx.x, lane = t % 64, wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int n0 = blockIdx.x * cols, r0 = blockIdx.y * RA;
  const int n_end = n0 + cols < N ? n0 + cols : N;
  const int fr = lane % 16, quad = lane / 16;
  const int l_row = lane / 32, l_kk = lane % 32;                       // a load: row l_row of 2, piece l_kk
  f32x4_t* const a_lds = gf_stage[wave];
  f32x4_t* const w_lds = gf_stage[wave] + P * RA * 32;
  const float* pa[LA];
  const float* pw[LW];
#pragma unroll
  for (int i = 0; i < LA; ++i) pa[i] = a + (size_t)(r0 + i * 2 + l_row < M ? r0 + i * 2 + l_row : r0) * lda;
#pragma unroll
  for (int i = 0; i < LW; ++i) pw[i] = w + (size_t)(n0 + i * 2 + l_row < n_end ? n0 + i * 2 + l_row : n0) * ldw;
  struct Set { f32x4_t a[P][LA], w[P][LW]; };
  f32x4_t gain[LN ? P : 1], add[LN ? P : 1];
  auto fetch = [&](Set& x, int set) {                                  // (past K: the row's first piece, dropped when it is parked)
    if constexpr (LN) {                                                // in the order of their use
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = (set * P + p) * GF_CHUNK + l_kk * 4, ks = k < K ? k : 0;
#pragma unroll
        for (int i = 0; i < LA; ++i) x.a[p][i] = *(const f32x4_t*)(pa[i] + ks);
      }
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = (set * P + p) * GF_CHUNK + l_kk * 4, ks = k < K ? k : 0;
        gain[p] = *(const f32x4_t*)(norm.g + ks);
        add[p] = *(const f32x4_t*)((norm.b ? norm.b : norm.g) + ks);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int k = (set * P + p) * GF_CHUNK + l_kk * 4, ks = k < K ? k : 0;
      if constexpr (!LN) {
#pragma unroll
        for (int i = 0; i < LA; ++i) x.a[p][i] = *(const f32x4_t*)(pa[i] + ks);
      }
#pragma unroll
      for (int i = 0; i < LW; ++i) x.w[p][i] = *(const f32x4_t*)(pw[i] + ks);
    }
  };
  // this lane's row of a fragment of a and of w, and the pieces of k group `quad` of it
  const int fp = fr / S, fs = fr % S;
  const int row_a = fp * RA + (fs & (RA - 1)), row_w = fp * CW + (fs < CW ? fs : 0);
  auto products = [&](Set& x, int set) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const bool in = (set * P + p) * GF_CHUNK + l_kk * 4 < K;
      const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < LA; ++i) a_lds[gf_place(p * RA + i * 2 + l_row, l_kk)] = in ? x.a[p][i] : zero;
#pragma unroll
      for (int i = 0; i < LW; ++i) w_lds[gf_place(p * CW + i * 2 + l_row, l_kk)] = in ? x.w[p][i] : zero;
    }
    gf_wave_order();
    floatx4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const f32x4_t fa = a_lds[gf_place(row_a, g * 4 + quad)], fw = w_lds[gf_place(row_w, g * 4 + quad)];
#pragma unroll
      for (int e = 0; e < 4; ++e) part = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fw[e], part, 0, 0, 0);
    }
    gf_wave_order();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 4 * quad + r, c = set * P + fp;
      if (i / S == fp && i % S < RA && fs < CW && c < n_chunks) gf_red[(c * RA + i % S) * (CW + 1) + fs] = part[r];
    }
  };
  const int n_sets = (n_chunks + P - 1) / P;
  Set x, y;
  int set = wave;
  if (set < n_sets) fetch(x, set);
  // what the epilogue needs is asked for behind the first operands, from places that always exist
  const int em = r0 + t / CW, en = n0 + t % CW;
  const bool e_ok = t < RA * CW && em < M && en < n_end;
  GF_EPILOGUE_LOADS
  if constexpr (LN) {
    // a row's 16 sums over 16 lanes (two a chunk), of the entries and then of the squares around the mean
    __builtin_amdgcn_sched_barrier(0);
    __shared__ __attribute__((aligned(16))) float gf_stat[2][RA][16];
    const bool on = set < n_sets;
    if (t < RA * 16 && t % 16 >= 2 * P * n_sets) gf_stat[0][t / 16][t % 16] = gf_stat[1][t / 16][t % 16] = 0.f;      // chunks that no wavefront has
    auto row_total = [&](int which, int row) {
      const f32x4_t* q = (const f32x4_t*)gf_stat[which][row];
      float s4[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) s4[j] = (q[j][0] + q[j][1]) + (q[j][2] + q[j][3]);
      return (s4[0] + s4[1]) + (s4[2] + s4[3]);
    };
    auto leave = [&](int which, int p, int i, float sum) {
      sum = group_sum<16>(sum);
      if (lane % 16 == 0) gf_stat[which][i * 2 + l_row][2 * (set * P + p) + l_kk / 16] = sum;
    };
    if (on) {
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int i = 0; i < LA; ++i) {
          const f32x4_t& v = x.a[p][i];
          leave(0, p, i, (set * P + p) * GF_CHUNK + l_kk * 4 < K ? (v[0] + v[1]) + (v[2] + v[3]) : 0.f);
        }
    }
    lds_barrier();
    if (on) {
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        const float mean = row_total(0, i * 2 + l_row) / (float)K;
#pragma unroll
        for (int p = 0; p < P; ++p) {
          f32x4_t& v = x.a[p][i];
          v -= mean;
          leave(1, p, i, (set * P + p) * GF_CHUNK + l_kk * 4 < K ? norm_squares(make_float4(v[0], v[1], v[2], v[3])) : 0.f);
        }
      }
    }
    lds_barrier();
    if (on) {
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        const float inv = 1.0f / sqrtf(row_total(1, i * 2 + l_row) / (float)K + norm.eps);
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) x.a[p][i][e] = norm_scaled(x.a[p][i][e], inv, gain[p][e], norm.b ? add[p][e] : 0.f);
      }
      products(x, set);
    }
  } else
  for (; set < n_sets; set += 2 * NW) {
    if (set + NW < n_sets) fetch(y, set + NW);
    products(x, set);
    if (set + 2 * NW < n_sets) fetch(x, set + 2 * NW);
    if (set + NW < n_sets) products(y, set + NW);
  }
  lds_barrier();
  if (!e_ok) return;
  const float* mine = gf_red + (t / CW) * (CW + 1) + t % CW;
  float v = mine[0];
#pragma unroll 4
  for (int c = 1; c < n_chunks; ++c) v += mine[c * RA * (CW + 1)];
  v = apply_act(v + e_bias_raw, ep.act);
  float* o = (float*)ep.out + (size_t)em * ep.ldo + en;
  *o = ep.accumulate ? e_old + v : v;
  if (kv.cache) kv_column_store<float>(kv, e_col, e_slot, v);
}

template <int WL, int AL, int NW, int CAP>
__global__ void __launch_bounds__(NW * 64)
gemm_f32_rows_kernel(const float* __restrict__ a, const float* __restrict__ w, void* out, int lda, int ldw, int ldo, int M, int N, int K,
                     int n_chunks, int cols, const void* bias, EpilogueRest er, KvScatter kv) {
  const Epilogue ep{bias, er.bias_dtype, er.act, er.accumulate, out, DA_F32, ldo};
  gemm_f32_rows_body<WL, AL, NW, CAP, false>(a, w, lda, ldw, M, N, K, n_chunks, cols, ep, kv, GfNorm{});
}
template <int WL, int AL, int NW>
__global__ void __launch_bounds__(NW * 64)
gemm_f32_ln_rows_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ g, const float* __restrict__ b, int ldw,
                        int M, int N, int K, int cols, float eps, void* out, int ldo, const void* bias, EpilogueRest er, KvScatter kv) {
  const Epilogue ep{bias, er.bias_dtype, er.act, er.accumulate, out, DA_F32, ldo};
  gemm_f32_rows_body<WL, AL, NW, GF_LN_MAX_K / GF_CHUNK, true>(x, w, K, ldw, M, N, K, (K + GF_CHUNK - 1) / GF_CHUNK, cols, ep, kv, GfNorm{g, b, eps});
}

// ---------------------------------------------------------------------------------------------
// Few rows, fragments straight from memory (16 rows x 64 bytes a load), a chunk a wavefront: 16 rows and 16, 8 or 4 columns a
// workgroup (the fewer, the fewer the products of 16 x 16 are; a fragment of w then holds its columns several times and the copies'
// results are dropped).  The loads are half cache lines, but a product starts with its first fragment, nothing waits for LDS, and
// four to twelve wavefronts that need little of it leave room for other workgroups.  Bound by the latency of its few loads at short
// k, else by half lines.
// ---------------------------------------------------------------------------------------------
template <int COLS, int NW, int CAP>
__global__ void __launch_bounds__(NW * 64)
gemm_f32_rows_direct_kernel(const float* __restrict__ a, const float* __restrict__ w, void* out, int lda, int ldw, int ldo, int M, int N, int K,
                            int n_chunks, const void* bias, EpilogueRest er, KvScatter kv) {
  const Epilogue ep{bias, er.bias_dtype, er.act, er.accumulate, out, DA_F32, ldo};
  __shared__ float gf_red[CAP * 16 * (COLS + 1)];               // [n_chunks][16][COLS + 1]
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int n0 = blockIdx.x * COLS, r0 = blockIdx.y * 16;
  const int fr = lane % 16, kq = (lane / 16) * 4;
  const float* pa = a + (size_t)(r0 + fr < M ? r0 + fr : r0) * lda;
  const float* pw = w + (size_t)(n0 + fr % COLS < N ? n0 + fr % COLS : n0) * ldw;
  // what the epilogue needs is asked for first, from places that always exist (a wavefront has one chunk, so there is no place behind
  // its first operands)
  const int em = r0 + t / COLS, en = n0 + t % COLS;
  const bool e_ok = t < 16 * COLS && em < M && en < N;
  GF_EPILOGUE_LOADS

  auto chunk = [&](int c, auto cutc) {
    constexpr bool CUT = decltype(cutc)::value;                        // the chunk that K cuts
    float4 av[8], wv[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      const int k = c * GF_CHUNK + g * 16 + kq, ks = (!CUT || k < K) ? k : 0;      // past K: the row's first piece, dropped
      av[g] = gf_load(pa + ks);
      wv[g] = gf_load(pw + ks);
    }
    floatx4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (CUT && c * GF_CHUNK + g * 16 + kq >= K) av[g] = wv[g] = make_float4(0.f, 0.f, 0.f, 0.f);
      part = gf_group(av[g], wv[g], part);
    }
    if (COLS == 16 || fr < COLS) {
#pragma unroll
      for (int r = 0; r < 4; ++r) gf_red[(c * 16 + 4 * (lane / 16) + r) * (COLS + 1) + fr] = part[r];
    }
  };
  const int whole = K / GF_CHUNK;
  for (int c = wave; c < n_chunks; c += NW) {
    if (c < whole) chunk(c, std::false_type{});
    else chunk(c, std::true_type{});
  }
  lds_barrier();
  if (!e_ok) return;
  const float* mine = gf_red + (t / COLS) * (COLS + 1) + t % COLS;
  float v = mine[0];
#pragma unroll 4
  for (int c = 1; c < n_chunks; ++c) v += mine[c * 16 * (COLS + 1)];
  v = apply_act(v + e_bias_raw, ep.act);
  float* o = (float*)ep.out + (size_t)em * ep.ldo + en;
  *o = ep.accumulate ? e_old + v : v;
  if (kv.cache) kv_column_store<float>(kv, e_col, e_slot, v);
}

// ---------------------------------------------------------------------------------------------
// Block tile BM x BN, WM x WN wavefronts.
// ---------------------------------------------------------------------------------------------
template <int BM, int BN, bool KTAIL>
__device__ __forceinline__ void
gemm_f32_tile_body(const float* __restrict__ a, int lda, const float* __restrict__ w, int ldw, const Epilogue& ep, const KvScatter& kv,
                   int M, int N, int K, int tiles_m, int tiles_n, float* smem) {
  constexpr int WM = 2, WN = 2, PF = 4, THREADS = WM * WN * 64;       // 2 x 2 wavefronts; slabs in flight
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int CA = BM * 8 / THREADS, CW = BN * 8 / THREADS;          // 16-byte pieces a thread and slab
  static_assert(BM * 8 % THREADS == 0 && BN * 8 % THREADS == 0, "the tile does not split over the threads");
  static_assert(GF_CHUNK == PF * GF_BK, "a chunk is a round of slabs");
  float* const As = smem;                                              // [2][BM][GF_LD]
  float* const Ws = smem + 2 * BM * GF_LD;                             // [2][BN][GF_LD]

  // Workgroups that follow each other in launch order land on different XCDs: each XCD takes a contiguous run of tiles,
  // m fastest, so that its workgroups share slabs of w in its L2.
  const int nblocks = tiles_m * tiles_n;
  int pid = blockIdx.x;
  {
    const int per = nblocks / 8, rem = nblocks % 8, xcd = pid % 8, local = pid / 8;
    pid = xcd * per + (xcd < rem ? xcd : rem) + local;
  }
  const int m0 = (pid % tiles_m) * BM, n0 = (pid / tiles_m) * BN;
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
  const int fr = lane % 16, kq = (lane / 16) * 4;
  const int kc = (t % 8) * 4;                                          // this thread's piece of a slab

  float4 ra[PF][CA], rw[PF][CW];
  const float* pa[CA];
  const float* pw[CW];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int row = m0 + (t + THREADS * i) / 8;
    pa[i] = a + (size_t)(row < M ? row : M - 1) * lda;
  }
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int row = n0 + (t + THREADS * i) / 8;
    pw[i] = w + (size_t)(row < N ? row : N - 1) * ldw;
  }
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  // (no conditional loads: pieces past K read the row's first piece and are replaced by zero)
#define GF_FETCH(stage, k0)                                                   \
  {                                                                           \
    const int k_ = (k0) + kc;                                                 \
    const bool in_ = !KTAIL || k_ < K;                                        \
    const int ks_ = in_ ? k_ : 0;                                             \
    _Pragma("unroll") for (int i = 0; i < CA; ++i) ra[stage][i] = gf_load(pa[i] + ks_); \
    _Pragma("unroll") for (int i = 0; i < CW; ++i) rw[stage][i] = gf_load(pw[i] + ks_); \
    if (KTAIL && !in_) {                                                      \
      _Pragma("unroll") for (int i = 0; i < CA; ++i) ra[stage][i] = zero;     \
      _Pragma("unroll") for (int i = 0; i < CW; ++i) rw[stage][i] = zero;     \
    }                                                                         \
  }
#define GF_STASH(stage, buf)                                                                                                  \
  {                                                                                                                           \
    _Pragma("unroll") for (int i = 0; i < CA; ++i) *(float4*)&As[((buf) * BM + (t + THREADS * i) / 8) * GF_LD + kc] = ra[stage][i]; \
    _Pragma("unroll") for (int i = 0; i < CW; ++i) *(float4*)&Ws[((buf) * BN + (t + THREADS * i) / 8) * GF_LD + kc] = rw[stage][i]; \
  }
  floatx4 acc[TM][TN], part[TM][TN];
  const floatx4 fzero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = part[i][j] = fzero;
  const int nslab = (K + GF_BK - 1) / GF_BK;
#pragma unroll
  for (int j = 0; j < PF; ++j)
    if (j < nslab) GF_FETCH(j, j * GF_BK);
  // What the epilogue needs, from places that always exist: behind the first slabs where there is a register for it (32 x 32: 5 of them; asked
  // for behind the products it was a round trip at the end of each tile: 526 x 3,072 x 768 38.9 -> 35.1 us, 526 x 768 x 768 14.3 -> 13.3), else before anything is stored.
  constexpr bool EARLY = TM * TN == 1;
  float bias[TN], old[TN][TM][4];
  auto ask = [&](int j) {
    const int n = n0 + wn + j * 16 + fr;
    const bool n_ok = n < N;
    bias[j] = (n_ok && ep.bias) ? load_param(ep.bias, ep.bias_dtype, n) : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + 4 * (lane / 16) + r;
        old[j][i][r] = *(n_ok && m < M && ep.accumulate ? (const float*)ep.out + (size_t)m * ep.ldo + n : w);
      }
  };
  if (EARLY) {
    da_read_arg(ep.act);
    ask(0);
  }
  GF_STASH(0, 0);
  lds_barrier();
  // Slab s: its registers (stage s % PF) went to LDS buffer s & 1 before the last barrier and take the slab PF further
  // on; the next slab's registers go to the other buffer, which was last read before the previous barrier.
#define GF_STEP(j, s, want_fetch, want_stash)                                                               \
  {                                                                                                         \
    constexpr int buf = (j) & 1;                                                                            \
    if (want_fetch) GF_FETCH(j, ((s) + PF) * GF_BK);                                                        \
    _Pragma("unroll") for (int kk = 0; kk < GF_BK; kk += 16) {                                              \
      float4 fa[TM], fw[TN];                                                                                \
      _Pragma("unroll") for (int i = 0; i < TM; ++i) fa[i] = *(const float4*)&As[(buf * BM + wm + i * 16 + fr) * GF_LD + kk + kq]; \
      _Pragma("unroll") for (int jj = 0; jj < TN; ++jj) fw[jj] = *(const float4*)&Ws[(buf * BN + wn + jj * 16 + fr) * GF_LD + kk + kq]; \
      _Pragma("unroll") for (int e = 0; e < 4; ++e)                                                         \
        _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                      \
          _Pragma("unroll") for (int jj = 0; jj < TN; ++jj)                                                 \
            part[i][jj] = __builtin_amdgcn_mfma_f32_16x16x4f32((&fa[i].x)[e], (&fw[jj].x)[e], part[i][jj], 0, 0, 0); \
    }                                                                                                       \
    if (want_stash) GF_STASH(((j) + 1) % PF, buf ^ 1);                                                      \
    lds_barrier();                                                                                          \
  }
#define GF_JOIN()                                              \
  _Pragma("unroll") for (int i = 0; i < TM; ++i)               \
    _Pragma("unroll") for (int jj = 0; jj < TN; ++jj) {        \
      acc[i][jj] += part[i][jj];                               \
      part[i][jj] = fzero;                                     \
    }
  int base = 0;
  for (; base + 2 * PF <= nslab; base += PF) {
    GF_STEP(0, base, true, true);
    GF_STEP(1, base + 1, true, true);
    GF_STEP(2, base + 2, true, true);
    GF_STEP(3, base + 3, true, true);
    GF_JOIN();
  }
  for (; base < nslab; base += PF) {
    if (base < nslab) GF_STEP(0, base, base + PF < nslab, base + 1 < nslab);
    if (base + 1 < nslab) GF_STEP(1, base + 1, base + 1 + PF < nslab, base + 2 < nslab);
    if (base + 2 < nslab) GF_STEP(2, base + 2, base + 2 + PF < nslab, base + 3 < nslab);
    if (base + 3 < nslab) GF_STEP(3, base + 3, base + 3 + PF < nslab, base + 4 < nslab);
    GF_JOIN();
  }
#undef GF_STEP
#undef GF_FETCH
#undef GF_STASH
#undef GF_JOIN

  // A lane holds column l % 16 and rows 4 * (l / 16) + r of each 16 x 16 piece: 64 consecutive bytes a row and store.
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 16 + fr;
    if (!EARLY) ask(j);
    KvColumn col;
    int slot[TM][4];                         // (the places in the cache only now: 32 x 32 would hold one workgroup fewer a compute unit)
    if (kv.cache) {
      col = kv_column(kv, n);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm + i * 16 + 4 * (lane / 16) + r;
          slot[i][r] = *(n < N && m < M ? kv.slot_map + m : (const int*)w);
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + 4 * (lane / 16) + r;
        if (n >= N || m >= M) continue;
        const float v = apply_act(acc[i][j][r] + bias[j], ep.act);
        ((float*)ep.out)[(size_t)m * ep.ldo + n] = ep.accumulate ? old[j][i][r] + v : v;
        if (kv.cache) kv_column_store<float>(kv, col, slot[i][r], v);
      }
  }
}

template <int BM, int BN>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ w, void* out, int lda, int ldw, int ldo, int M, int N, int K, int tiles_m,
                     int tiles_n, const void* bias, EpilogueRest er, KvScatter kv) {
  const Epilogue ep{bias, er.bias_dtype, er.act, er.accumulate, out, DA_F32, ldo};
  __shared__ __attribute__((aligned(16))) float smem[2 * (BM + BN) * GF_LD];
  if (K % GF_BK == 0) gemm_f32_tile_body<BM, BN, false>(a, lda, w, ldw, ep, kv, M, N, K, tiles_m, tiles_n, smem);
  else gemm_f32_tile_body<BM, BN, true>(a, lda, w, ldw, ep, kv, M, N, K, tiles_m, tiles_n, smem);
}

template <int BM, int BN>
static void launch_f32_tile(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                            int M, int N, int K) {
  const int tiles_m = da_ceil_div(M, BM), tiles_n = da_ceil_div(N, BN);
  hipLaunchKernelGGL((gemm_f32_tile_kernel<BM, BN>), dim3(tiles_m * tiles_n), dim3(256), 0, s, a, w, ep.out, lda, ldw, ep.ldo, M, N, K,
                     tiles_m, tiles_n, ep.bias, epilogue_rest(ep), kv);
}

template <int WL, int AL, int NW, int CAP>
static void launch_f32_rows(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                            int M, int N, int K, int cols) {
  hipLaunchKernelGGL((gemm_f32_rows_kernel<WL, AL, NW, CAP>), dim3(da_ceil_div(N, cols), da_ceil_div(M, 4 * AL)), dim3(NW * 64), 0, s, a, w,
                     ep.out, lda, ldw, ep.ldo, M, N, K, da_ceil_div(K, GF_CHUNK), cols, ep.bias, epilogue_rest(ep), kv);
}
// The wavefronts and the room for partial sums, by K.  More workgroups than compute units (16 columns each, then): few wavefronts
// each, so that several workgroups share a compute unit's LDS and one's loads run beside another's products (K = 768, N = 50,257: 4 rows
// 32 us with 3 wavefronts, 45 with 6; 8 rows 38 / 51; 32 rows, N = 3,072 7.9 with 4, 8.8 with 6).
template <int WL, int AL>
static void launch_f32_rows_k(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                              int M, int N, int K, int cols) {
  if constexpr (WL == 4) {
    if ((long)da_ceil_div(N, cols) * da_ceil_div(M, 4 * AL) > 256 && K <= (AL == 4 ? 8 : 24) * GF_CHUNK) {
      launch_f32_rows<WL, AL, AL == 4 ? 4 : 3, AL == 4 ? 8 : 24>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
      return;
    }
  }
  if (K <= 6 * GF_CHUNK) launch_f32_rows<WL, AL, 6, 6>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
  else if (K <= 24 * GF_CHUNK) launch_f32_rows<WL, AL, 8, 24>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
  else launch_f32_rows<WL, AL, AL == 4 ? 6 : 8, GF_ROWS_CAP>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
}
template <int AL>
static void launch_f32_rows_n(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                              int M, int N, int K, int cols) {
  if (cols <= 4) launch_f32_rows_k<1, AL>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
  else if (cols <= 8) launch_f32_rows_k<2, AL>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
  else if (cols <= 12) launch_f32_rows_k<3, AL>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
  else launch_f32_rows_k<4, AL>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
}

template <int COLS, int NW, int CAP>
static void launch_f32_rows_direct_k(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                                     int M, int N, int K) {
  hipLaunchKernelGGL((gemm_f32_rows_direct_kernel<COLS, NW, CAP>), dim3(da_ceil_div(N, COLS), da_ceil_div(M, 16)), dim3(NW * 64), 0, s, a, w,
                     ep.out, lda, ldw, ep.ldo, M, N, K, da_ceil_div(K, GF_CHUNK), ep.bias, epilogue_rest(ep), kv);
}
template <int COLS>
static void launch_f32_rows_direct(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                                   int M, int N, int K) {
  if (K <= 4 * GF_CHUNK) launch_f32_rows_direct_k<COLS, 4, 4>(s, a, lda, w, ldw, ep, kv, M, N, K);
  else if (K <= 8 * GF_CHUNK) launch_f32_rows_direct_k<COLS, 8, 8>(s, a, lda, w, ldw, ep, kv, M, N, K);
  else if (K <= 24 * GF_CHUNK) launch_f32_rows_direct_k<COLS, 12, 24>(s, a, lda, w, ldw, ep, kv, M, N, K);
  else launch_f32_rows_direct_k<COLS, 12, GF_ROWS_CAP>(s, a, lda, w, ldw, ep, kv, M, N, K);
}

enum { GF_AUTO = 0, GF_ROWS, GF_64x64, GF_32x32, GF_ROWS_DIRECT, GF_ROWS_STAGED, GF_LAST = GF_ROWS_STAGED };

// Which kernel a product goes to.  Measured on MI355X with K from 768 to 4,096:
//  - the kernel for few rows up to 8 rows (768 x 50,257: 4 rows 31 us against 38 in tiles of 32 x 32, 8 rows 38.1 against 38.4, 16
//    rows 46 against 38) and where its products of 16 x 16 are at most 512 (100 x 768 x 768 6.8 us against 9.8, 64 x 768 x 3,072
//    11.4 against 27, 32 x 3,072 x 768 7.9 against 10.9; with 528 of them, 170 x 768 x 768, 10.9 against 9.7);
//  - else tiles of 64 x 64 where there are 700 and more, counting what M and N waste of them (1,000 x 3,072 x 768 47 against
//    51 us, 526 x 50,257 x 768 392 against 400, but 200 x 50,257 x 768 183 against 167);
//  - else tiles of 32 x 32 (526 x 3,072 x 768, 432 of the larger tiles: 31 against 34 us).
static int f32_form(int M, int N, int K) {
  if (K <= GF_ROWS_MAX_K && (M <= 8 || (long)da_ceil_div(M, 16) * da_ceil_div(N, 16) <= 512)) return GF_ROWS;
  const long large = (long)da_ceil_div(M, 64) * da_ceil_div(N, 64), small = (long)da_ceil_div(M, 32) * da_ceil_div(N, 32);
  return large >= 700 && large * 40 <= small * 11 ? GF_64x64 : GF_32x32;      // (a small tile's share of the chip costs 10 % more)
}

// Which of the two kernels for few rows.  The staged one reads whole lines, and below about 208 products of 16 x 16 its columns are
// divided so that every compute unit has a workgroup; the direct one has the shorter chain, and more workgroups a compute unit.
// Measured over 7,190 sizes (K 256 to 6,400, N 64 to 50,257, M 1 to 256, cold weights), the rule takes 0.892 of the direct kernel's time in
// the mean, the better of the two 0.885; what it takes is at most 12 % (0.8 us) behind the direct kernel.  us, direct / staged:
//  - up to 3 chunks of k: direct (K = 256: 4 x 512 2.8 / 3.4, 8 x 9,216 5.4 / 6.1; K = 384: 8 x 11,264 6.2 / 7.3);
//  - 25 rows and more: staged (K = 768: 100 x 768 7.7 / 6.6; K = 3,072: 48 x 2,304 26 / 22), but for 33 to 40 rows, whose last 16 are mostly
//    padding, with 9 to 13 chunks (wavefronts of the staged kernel left over) and up to 400 products (K = 1,152: 33 x 2,048 9.7 / 10.9);
//  - 17 to 24 rows: staged up to 256 products (K = 3,072: 17 x 1,920 13.6 / 12.1), direct above (17 x 2,304 17.0 / 19.8);
//  - up to 16 rows and 208 products: staged (4 rows, K = 768 x 768 4.4 / 3.6; K = 4,096 x 1,024 13.3 / 6.6), but direct up to 12 rows with 9 to 13
//    chunks and more than 128 products (K = 1,152, 4 x 3,072 6.0 / 6.5);
//  - up to 16 rows and more products: a second round of workgroups begins.  13 to 16 rows: staged from 14 chunks on (K = 5,120, 16 x 4,800
//    48 / 37; K = 1,152 16 x 6,144 12.1 / 13.4).  Up to 12 rows: staged from 40 chunks on (K = 6,400, 8 x 6,144 46.7 / 42.7), and up to 8 rows with 4
//    or 14 to 16 chunks and up to 256 products, with 14 to 20 chunks (K = 1,920, 8 x 5,120 17.4 / 14.0), and for vocabularies (K = 768, 4 x 50,257
//    39 / 31); else direct (K = 768, 4 x 6,144 6.8 / 7.9; K = 1,024, 4 x 4,100 6.8 / 8.6; K = 4,096, 4 x 8,192 29.8 / 33.9).
static bool f32_rows_staged(int M, int N, int K) {
  const int chunks = da_ceil_div(K, GF_CHUNK);
  const long products = (long)da_ceil_div(M, 16) * da_ceil_div(N, 16);
  const bool left_over = chunks >= 9 && chunks <= 13;
  if (chunks <= 3) return false;
  if (M > 24) return !(left_over && M > 32 && M <= 40 && products > 176 && products <= 400);
  if (M > 16) return products <= 256;
  if (products <= 208) return M > 12 || !(left_over && products > 128);
  if (M > 12) return chunks > 13;
  if (chunks >= 40) return true;
  if (M > 8) return false;
  if (products <= 256) return chunks == 4 || (chunks >= 14 && chunks <= 16);
  if (chunks >= 14) return chunks <= 20 || (chunks <= 24 && N >= 16384);
  return N >= (chunks >= 9 ? 16384 : 32000) && chunks >= 5;
}

// The columns a workgroup of the staged kernel: every compute unit a workgroup, and no second round of them for less than 16
// columns (48 x 1,024, K = 1,600: 13 columns in 79 x 3 workgroups 8.8 us, 12 in 86 x 3 13.0; direct 8.3).
static int f32_rows_columns(int M, int N) {
  const int blocks = da_ceil_div(M, M <= 4 ? 4 : (M <= 8 ? 8 : 16)), share = da_ceil_div(N, blocks < 256 ? 256 / blocks : 1);
  return share > 16 ? 16 : share;
}
// 0 where a product of few rows goes to the direct kernel, else the columns a workgroup of the staged one.
extern "C" int da_gemm_f32_rows_choice(int M, int N, int K) { return f32_rows_staged(M, N, K) ? f32_rows_columns(M, N) : 0; }

// Whether a LayerNorm and the product behind it are one kernel: up to 8 rows and GF_LN_MAX_K columns of the stream (the sizes whose norm alone
// is layernorm_row_kernel<1, 4>) where that is ahead.  Every workgroup normalises all rows, so the rows count; a launch less is worth 1.6 us.
// us, cold weights, the two kernels / this, 4 and 8 rows:
//   K = 768:   N = 64 5.6 / 5.0, 5.6 / 5.7; 1,100 5.8 / 4.9, 6.1 / 6.0; 2,304 6.7 / 5.7, 6.8 / 6.7; 3,072 7.0 / 5.9, 7.1 / 6.7; 4,096 7.7 / 6.3, 7.8 / 7.3
//   K = 1,024: N = 768 5.9 / 5.3, 6.2 / 6.3; 3,072 7.4 / 6.4, 7.6 / 7.4; 3,600 7.9 / 6.8, 8.0 / 7.9; 4,096 7.8 / 7.4, 8.0 / 8.5
//   K = 256:   N = 500 5.3 / 4.9, 5.6 / 5.4; 3,072 6.0 / 4.1, 6.0 / 5.0;  K = 64: N = 500 4.7 / 4.8, 4.7 / 5.3; 2,000 4.7 / 4.2, 4.7 / 5.1; 3,100 5.0 / 3.9, 5.0 / 4.8
// (1 row: 6.2 / 5.6 at K = 768, N = 2,304, 4.2 / 4.8 at K = 64, N = 500.)  More than 4,096 columns are a second round of workgroups.
extern "C" int da_gemm_f32_ln_takes(int M, int N, int K) {
  if (M < 1 || M > 8 || K < 1 || K > GF_LN_MAX_K || K % 4 || N < 1 || N > 4096) return 0;
  if (M <= 4) return K >= 128 || N > 1024;
  return K >= 128 && N > 1024 && (K <= 896 || N <= 3600);
}

template <int AL, int NW>
static void launch_f32_ln_rows(hipStream_t s, const float* x, const float* w, const float* g, const float* b, float eps, int ldw, const Epilogue& ep,
                               const KvScatter& kv, int M, int N, int K) {
  const int cols = f32_rows_columns(M, N);
#define GF_LN_GO(WL)                                                                                                                          \
  hipLaunchKernelGGL((gemm_f32_ln_rows_kernel<WL, AL, NW>), dim3(da_ceil_div(N, cols)), dim3(NW * 64), 0, s, x, w, g, b, ldw, M, N, K, cols, eps, \
                     ep.out, ep.ldo, ep.bias, epilogue_rest(ep), kv)
  if (cols <= 4) GF_LN_GO(1);
  else if (cols <= 8) GF_LN_GO(2);
  else if (cols <= 12) GF_LN_GO(3);
  else GF_LN_GO(4);
#undef GF_LN_GO
}
// out = act(LayerNorm(x) @ w.T + bias): x's rows K apart, gain and bias of the norm 32-bit (b may be null).
extern "C" int da_gemm_f32_ln(const float* x, const float* g, const float* b, float eps, const float* w, int ldw, const void* bias, int bias_dtype,
                              int act, float* out, int ldo, int M, int N, int K, float* kv_cache, const int* slot_map, int q_cols, int kv_cols,
                              int Hkv, int D, int page, void* stream) {
  DA_REQUIRE(M >= 0 && N > 0 && K > 0 && eps > 0.f, "gemm_f32_ln: bad sizes M=%d N=%d K=%d eps=%g", M, N, K, eps);
  DA_REQUIRE(ldw % 4 == 0 && ldw >= K && ldo >= N, "gemm_f32_ln: row lengths (ldw=%d ldo=%d)", ldw, ldo);
  DA_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)g % 16 == 0 && (uintptr_t)b % 16 == 0,
             "gemm_f32_ln: operands, gain and bias must be 16-byte aligned");
  DA_REQUIRE(act >= DA_ACT_NONE && act <= DA_ACT_LAST, "gemm_f32_ln: unknown activation %d", act);
  if (kv_cache) {
    DA_REQUIRE(slot_map && q_cols >= 0 && kv_cols == Hkv * D && q_cols + 2 * kv_cols == N && page > 0,
               "gemm_f32_ln: the q|k|v columns (%d + 2*%d) must add up to N=%d", q_cols, kv_cols, N);
  }
  if (M == 0) return 0;
  DA_REQUIRE(da_gemm_f32_ln_takes(M, N, K), "gemm_f32_ln: %d rows, %d columns, K=%d are not taken", M, N, K);
  const Epilogue ep{bias, bias_dtype, act, 0, out, DA_F32, ldo};
  const KvScatter kv{kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page};
  hipStream_t s = (hipStream_t)stream;
  const bool six = K <= 6 * GF_CHUNK;                      // (a set a wavefront)
  if (M <= 4) { if (six) launch_f32_ln_rows<1, 6>(s, x, w, g, b, eps, ldw, ep, kv, M, N, K); else launch_f32_ln_rows<1, 8>(s, x, w, g, b, eps, ldw, ep, kv, M, N, K); }
  else { if (six) launch_f32_ln_rows<2, 6>(s, x, w, g, b, eps, ldw, ep, kv, M, N, K); else launch_f32_ln_rows<2, 8>(s, x, w, g, b, eps, ldw, ep, kv, M, N, K); }
  DA_CHECK_LAUNCH("gemm_f32_ln");
  return 0;
}

// out (+)= act(a @ w.T + bias).  `form` 0: chosen by the sizes; else that kernel (tests and timing), where it takes them.
extern "C" int da_gemm_f32(const float* a, int lda, const float* w, int ldw, const void* bias, int bias_dtype, int act, int accumulate,
                           float* out, int ldo, int M, int N, int K, float* kv_cache, const int* slot_map, int q_cols, int kv_cols,
                           int Hkv, int D, int page, int form, void* stream) {
  DA_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  DA_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0, "gemm_f32: K, lda and ldw must be multiples of 4 (K=%d lda=%d ldw=%d)", K, lda, ldw);
  DA_REQUIRE((uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0, "gemm_f32: operands must be 16-byte aligned");
  DA_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm_f32: leading sizes too small (lda=%d ldw=%d ldo=%d)", lda, ldw, ldo);
  DA_REQUIRE(act >= DA_ACT_NONE && act <= DA_ACT_LAST, "gemm_f32: unknown activation %d", act);
  DA_REQUIRE(form >= GF_AUTO && form <= GF_LAST, "gemm_f32: unknown form %d", form);
  DA_REQUIRE(form == GF_AUTO || form == GF_64x64 || form == GF_32x32 || K <= GF_ROWS_MAX_K, "gemm_f32: the kernel for few rows takes K up to %d (K=%d)", GF_ROWS_MAX_K, K);
  if (kv_cache) {
    DA_REQUIRE(!accumulate && slot_map && q_cols >= 0 && kv_cols == Hkv * D && q_cols + 2 * kv_cols == N && page > 0,
               "gemm_f32: the q|k|v columns (%d + 2*%d) must add up to N=%d", q_cols, kv_cols, N);
  }
  if (M == 0) return 0;
  const Epilogue ep{bias, bias_dtype, act, accumulate, out, DA_F32, ldo};
  const KvScatter kv{kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page};
  hipStream_t s = (hipStream_t)stream;
  if (form == GF_AUTO) form = f32_form(M, N, K);
  if (form == GF_ROWS) form = f32_rows_staged(M, N, K) ? GF_ROWS_STAGED : GF_ROWS_DIRECT;
  switch (form) {
    case GF_ROWS_DIRECT: {
      const long tiles = (long)da_ceil_div(M, 16) * da_ceil_div(N, 16);
      if (tiles <= 64) launch_f32_rows_direct<4>(s, a, lda, w, ldw, ep, kv, M, N, K);
      else if (tiles <= 128) launch_f32_rows_direct<8>(s, a, lda, w, ldw, ep, kv, M, N, K);
      else launch_f32_rows_direct<16>(s, a, lda, w, ldw, ep, kv, M, N, K);
      break;
    }
    case GF_ROWS_STAGED: {
      const int cols = f32_rows_columns(M, N);
      if (M <= 4) launch_f32_rows_n<1>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
      else if (M <= 8) launch_f32_rows_n<2>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
      else launch_f32_rows_n<4>(s, a, lda, w, ldw, ep, kv, M, N, K, cols);
      break;
    }
    case GF_64x64: launch_f32_tile<64, 64>(s, a, lda, w, ldw, ep, kv, M, N, K); break;
    default: launch_f32_tile<32, 32>(s, a, lda, w, ldw, ep, kv, M, N, K); break;
  }
  DA_CHECK_LAUNCH("gemm_f32");
  return 0;
}
