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
//  * gemm_f32_rows: few rows.  A workgroup owns 16 rows and up to 16 columns; its wavefronts take whole chunks, straight
//    from memory into fragments, and the chunks' sums are added through LDS.  Bound by the bytes of w.
//  * gemm_f32_tile: block tiles of 64 x 64 or 32 x 32 through two LDS buffers, slabs of 32 k, the next four slabs in flight
//    in registers.  Bound by the matrix cores (157 TFLOP/s in 32-bit) where the tiles fill the chip several times over:
//    1,000 x 50,257 x 768 in 687 us, 72 % of that rate; below, by the latency of a slab, which small tiles, several of
//    them on a compute unit, hide better than large ones (526 x 3,072 x 768: 32 x 32 31 us, 64 x 64 34, 128 x 128 72).
//
// Measured on MI355X beside the plain kernel (gemm_ref.hip), which a product of 4 rows walks in 64 x 64 tiles through one
// LDS buffer: 4 x 768 x 3,072 226 -> 10 us, 4 x 2,304 x 768 86 -> 4.4, 526 x 768 x 3,072 about 360 -> 37,
// 526 x 2,304 x 768 128 -> 24, 526 x 50,257 x 768 1,308 -> 384.
#include "gemm_common.h"
#include <type_traits>

#define GF_CHUNK 128
#define GF_BK 32
#define GF_LD (GF_BK + 4)    // padded LDS row, floats (144 bytes): 16 consecutive rows start in different banks

__device__ __forceinline__ float4 gf_load(const float* p) { return *(const float4*)p; }
__device__ __forceinline__ floatx4 gf_group(const float4& a, const float4& w, floatx4 c) {      // the 16 k of a group
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, w.x, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, w.y, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, w.z, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, w.w, c, 0, 0, 0);
}

// the k and v columns of a q|k|v product (column n >= q_cols of the row whose place in the cache is `slot`)
__device__ __forceinline__ void gf_scatter(const KvScatter& kv, int slot, int n, float v) {
  const int pg = slot / kv.page, row = slot % kv.page;
  const int c2 = n - kv.q_cols, is_v = c2 >= kv.kv_cols, cc = is_v ? c2 - kv.kv_cols : c2;
  const int h = cc / kv.D, d = cc % kv.D;
  float* cache = (float*)kv.cache;
  if (is_v) cache[cache_v_base(pg, h, kv.Hkv, kv.page, kv.D) + (long long)d * kv.page + row] = v;
  else cache[cache_k_row(pg, h, row, kv.Hkv, kv.page, kv.D) + d] = v;
}

// ---------------------------------------------------------------------------------------------
// Few rows: blockIdx.x: COLS columns (16, or 8 or 4 where the columns alone would leave compute units idle: the
// fragment of w then holds them several times and the copies' results are dropped), blockIdx.y: 16 rows.
// ---------------------------------------------------------------------------------------------
// CAP: chunks that the partial sums in LDS have room for.
template <int COLS, int NW, int CAP>
__global__ void __launch_bounds__(NW * 64)
gemm_f32_rows_kernel(const float* __restrict__ a, int lda, const float* __restrict__ w, int ldw, Epilogue ep, KvScatter kv,
                     int M, int N, int K, int n_chunks) {
  __shared__ float gf_red[CAP * 16 * (COLS + 1)];                      // [n_chunks][16][COLS + 1]
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int n0 = blockIdx.x * COLS, r0 = blockIdx.y * 16;
  const int fr = lane % 16, kq = (lane / 16) * 4;
  const float* pa = a + (size_t)(r0 + fr < M ? r0 + fr : r0) * lda;
  const float* pw = w + (size_t)(n0 + fr % COLS < N ? n0 + fr % COLS : n0) * ldw;
  // what the epilogue needs is asked for first, from places that always exist
  const int em = r0 + t / COLS, en = n0 + t % COLS;
  const bool e_ok = t < 16 * COLS && em < M && en < N;
  const float e_bias_raw = (e_ok && ep.bias) ? load_param(ep.bias, ep.bias_dtype, en) : 0.f;
  const float e_old = *((e_ok && ep.accumulate) ? (const float*)ep.out + (size_t)em * ep.ldo + en : w);
  const int e_slot = *((e_ok && kv.cache) ? kv.slot_map + em : (const int*)w);

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
  if (kv.cache && en >= kv.q_cols && e_slot >= 0) gf_scatter(kv, e_slot, en, v);
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
  // What += adds to is asked for before anything is stored, from places that always exist.
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 16 + fr;
    const bool n_ok = n < N;
    const float bias = (n_ok && ep.bias) ? load_param(ep.bias, ep.bias_dtype, n) : 0.f;
    float old[TM][4];
    int slot[TM][4];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + 4 * (lane / 16) + r;
        const bool ok = n_ok && m < M;
        old[i][r] = ep.accumulate ? *(ok ? (const float*)ep.out + (size_t)m * ep.ldo + n : w) : 0.f;
        slot[i][r] = kv.cache ? *(ok ? kv.slot_map + m : (const int*)w) : -1;
      }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + 4 * (lane / 16) + r;
        if (!n_ok || m >= M) continue;
        const float v = apply_act(acc[i][j][r] + bias, ep.act);
        ((float*)ep.out)[(size_t)m * ep.ldo + n] = ep.accumulate ? old[i][r] + v : v;
        if (kv.cache && n >= kv.q_cols && slot[i][r] >= 0) gf_scatter(kv, slot[i][r], n, v);
      }
  }
}

template <int BM, int BN>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(const float* __restrict__ a, int lda, const float* __restrict__ w, int ldw, Epilogue ep, KvScatter kv,
                     int M, int N, int K, int tiles_m, int tiles_n) {
  __shared__ __attribute__((aligned(16))) float smem[2 * (BM + BN) * GF_LD];
  if (K % GF_BK == 0) gemm_f32_tile_body<BM, BN, false>(a, lda, w, ldw, ep, kv, M, N, K, tiles_m, tiles_n, smem);
  else gemm_f32_tile_body<BM, BN, true>(a, lda, w, ldw, ep, kv, M, N, K, tiles_m, tiles_n, smem);
}

template <int BM, int BN>
static void launch_f32_tile(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                            int M, int N, int K) {
  const int tiles_m = da_ceil_div(M, BM), tiles_n = da_ceil_div(N, BN);
  hipLaunchKernelGGL((gemm_f32_tile_kernel<BM, BN>), dim3(tiles_m * tiles_n), dim3(256), 0, s, a, lda, w, ldw, ep, kv, M, N, K, tiles_m,
                     tiles_n);
}

template <int COLS, int NW, int CAP>
static void launch_f32_rows(hipStream_t s, const float* a, int lda, const float* w, int ldw, const Epilogue& ep, const KvScatter& kv,
                            int M, int N, int K) {
  hipLaunchKernelGGL((gemm_f32_rows_kernel<COLS, NW, CAP>), dim3(da_ceil_div(N, COLS), da_ceil_div(M, 16)), dim3(NW * 64), 0, s, a, lda,
                     w, ldw, ep, kv, M, N, K, da_ceil_div(K, GF_CHUNK));
}

enum { GF_AUTO = 0, GF_ROWS, GF_64x64, GF_32x32, GF_LAST = GF_32x32 };
#define GF_ROWS_CAP 50
#define GF_ROWS_MAX_K (GF_ROWS_CAP * GF_CHUNK)      // the chunks' sums of 16 x 16 outputs fit in 64 KB of LDS

// Which kernel a product goes to.  Measured on MI355X with K from 768 to 4,096:
//  - the kernel for few rows up to 8 rows (the head: 4 rows 30 against 32 us, 16 rows 39 against 32) and where its
//    workgroups are at most 512, which is what the chip runs side by side (64 x 768 x 3,072 13 against 26 us, 100 x 768 x 768
//    7.7 against 9.8, 32 x 3,072 x 768 8.0 against 10.3; with 576 of them 10.5 against 9.8);
//  - else tiles of 64 x 64 where there are 700 and more, counting what M and N waste of them (1,000 x 3,072 x 768 47 against
//    51 us, 526 x 50,257 x 768 384 against 401, but 200 x 50,257 x 768 183 against 167);
//  - else tiles of 32 x 32 (526 x 3,072 x 768, 432 of the larger tiles: 31 against 34 us).
static int f32_form(int M, int N, int K) {
  if (K <= GF_ROWS_MAX_K && (M <= 8 || (long)da_ceil_div(M, 16) * da_ceil_div(N, 16) <= 512)) return GF_ROWS;
  const long large = (long)da_ceil_div(M, 64) * da_ceil_div(N, 64), small = (long)da_ceil_div(M, 32) * da_ceil_div(N, 32);
  return large >= 700 && large * 40 <= small * 11 ? GF_64x64 : GF_32x32;      // (a small tile's share of the chip costs 10 % more)
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
  DA_REQUIRE(form != GF_ROWS || K <= GF_ROWS_MAX_K, "gemm_f32: the kernel for few rows takes K up to %d (K=%d)", GF_ROWS_MAX_K, K);
  if (kv_cache) {
    DA_REQUIRE(!accumulate && slot_map && q_cols >= 0 && kv_cols == Hkv * D && q_cols + 2 * kv_cols == N && page > 0,
               "gemm_f32: the q|k|v columns (%d + 2*%d) must add up to N=%d", q_cols, kv_cols, N);
  }
  if (M == 0) return 0;
  const Epilogue ep{bias, bias_dtype, act, accumulate, out, DA_F32, ldo};
  const KvScatter kv{kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page};
  hipStream_t s = (hipStream_t)stream;
  if (form == GF_AUTO) form = f32_form(M, N, K);
#define DA_GF_ROWS(C)                                                                                        \
  do {                                                                                                       \
    if (K <= 4 * GF_CHUNK) launch_f32_rows<C, 4, 4>(s, a, lda, w, ldw, ep, kv, M, N, K);                     \
    else if (K <= 8 * GF_CHUNK) launch_f32_rows<C, 8, 8>(s, a, lda, w, ldw, ep, kv, M, N, K);                \
    else if (K <= 24 * GF_CHUNK) launch_f32_rows<C, 12, 24>(s, a, lda, w, ldw, ep, kv, M, N, K);             \
    else launch_f32_rows<C, 12, GF_ROWS_CAP>(s, a, lda, w, ldw, ep, kv, M, N, K);                            \
  } while (0)
  switch (form) {
    case GF_ROWS: {
      const long tiles = (long)da_ceil_div(M, 16) * da_ceil_div(N, 16);
      if (tiles <= 64) DA_GF_ROWS(4);
      else if (tiles <= 128) DA_GF_ROWS(8);
      else DA_GF_ROWS(16);
      break;
    }
    case GF_64x64: launch_f32_tile<64, 64>(s, a, lda, w, ldw, ep, kv, M, N, K); break;
    default: launch_f32_tile<32, 32>(s, a, lda, w, ldw, ep, kv, M, N, K); break;
  }
#undef DA_GF_ROWS
  DA_CHECK_LAUNCH("gemm_f32");
  return 0;
}
