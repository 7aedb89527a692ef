// bfloat16 matrix products on the gfx950 matrix cores, with the epilogues a block needs:
//
//   out[m, n] (+)= act( sum_k a[m, k] * w[n, k] + bias[n] )
//
// a: [M, K] bf16, w: [N, K] bf16 ("[out, in]", K contiguous), 32-bit accumulation; out is bf16,
// or 32-bit (plain store or += for the residual stream).  Three kernels:
//
//  * gemm_tile: block tiles of 64x64 to 128x128 (MFMA 32x32x16), operands staged through two LDS
//    buffers, with the next four slabs already in flight in registers.  For steps with many rows
//    (prefill).  Products whose sizes suit them go to gemm_wide.hip's tiles instead (da_gemm_wide_choice).
//  * gemm_skinny: for M <= 64 (decode); gemm_skinny32 where they would be more workgroups than compute units (sk_one_a_unit).  A workgroup owns 16 output columns; its wavefronts (4 to 12)
//    split K, pull their part of a and w from memory in whole cache lines, pass it through LDS into
//    MFMA 16x16x32 fragments and add their sums through LDS in a fixed order.  Bound by the bytes of w.
//  * gemm_skinny4: for M <= 4 (8 with a long K) and up to 2,048 columns.  MFMA 16x16x32 with four pieces of k side by side, so that
//    four rows of w are read in whole cache lines straight into registers; 4 or 8 columns a workgroup.
//
// In each, an output element sums over k in an order that depends on K only, never on M or on
// the row's place in the batch.
//
// MFMA fragment layout (64 lanes).  32x32x16: lane l gives row (a) / column (b) l % 32 and the
// 8 consecutive k starting at 8 * (l / 32); it receives, for r in 0..15, the element at
// row 8 * (r / 4) + 4 * (l / 32) + r % 4, column l % 32.  16x16x32: lane l gives row / column
// l % 16 and k = 8 * (l / 16) .. +7; it receives rows 4 * (l / 16) + r, r in 0..3, column l % 16.
#include "gemm_common.h"
#include "gemm_skinny32.h"
#include <da_read_arg.h>      // (the simulator on the CPU has one of its own)
#include <type_traits>

#define BKT 64               // k per slab
#define LDS_LD (BKT + 8)     // padded row length in elements (144 bytes): spreads rows over banks

// ---------------------------------------------------------------------------------------------
// Block tile BM x BN, WM x WN wavefronts of (BM/WM) x (BN/WN) each.  Two LDS buffers: while slab k is
// multiplied out of one, the loads of slab k+1 are in flight and are then parked in the other; one
// barrier per slab.
// ---------------------------------------------------------------------------------------------
// OUTMODE: 0 bf16 store, 1 f32 store, 2 f32 +=.  ACT and OUTMODE are compile-time so that the
// epilogue is straight-line code.
// ---------------------------------------------------------------------------------------------
// The epilogue of a block tile.  A lane holds one column and 16 scattered rows of each 32 x 32 piece,
// two or four bytes wide: stored from there, a wavefront's store covers 64 bytes a row.  Instead the
// workgroup parks the tile in LDS (bias and activation applied, rounded to the output's type) and
// stores it row by row in 16-byte pieces, a whole row of the tile side by side; what += adds to is
// loaded the same way.  All loads come first and are used in straight-line code, only stores stand
// under conditions: a load under a condition would make each store wait for the one before it.
// OUTMODE: 0 bf16 store, 1 f32 store, 2 f32 +=.
// ---------------------------------------------------------------------------------------------
template <int BM, int BN, int OUTMODE>
constexpr int tile_out_bytes() {
  return BM * (BN + (OUTMODE == 0 ? 8 : 4)) * (OUTMODE == 0 ? 2 : 4);
}
// ... and behind it, for a fused q|k|v projection, the tile rows' places in the cache and how the values of each 32 rows go there
template <int BM, int OUTMODE>
constexpr int tile_slot_bytes() { return OUTMODE == 0 ? BM * 4 + BM / 32 * 4 : 0; }

template <int BM, int BN, int WM, int WN, int ACT, int OUTMODE>
__device__ __forceinline__ void
tile_epilogue(floatx16 (&acc)[BM / WM / 32][BN / WN / 32], const float (&bias)[BN / WN / 32], char* smem, const void* safe,
              const Epilogue& ep, const KvScatter& kv, int slot, int M, int N, int m0, int n0) {
  constexpr int THREADS = WM * WN * 64;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int ES = OUTMODE == 0 ? 2 : 4, CH = 16 / ES;      // bytes an element; elements a 16-byte piece
  constexpr int LDT = BN + CH;                                 // a parked row, padded by one piece
  constexpr int CPR = BN / CH, NCHK = BM * CPR / THREADS;      // pieces a row; pieces a thread
  static_assert(BM * CPR % THREADS == 0, "the tile's pieces do not split over the threads");
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
  const int fr = lane % 32;
  int* slots = (int*)(smem + tile_out_bytes<BM, BN, OUTMODE>());        // the tile rows' places, -1: none
  int* ways = slots + BM;                                               // of each 32 rows: KV_WAY_RUNS (kv_all_runs) or kv_run_offset
  const bool vwide = OUTMODE == 0 && kv.cache && (uintptr_t)kv.cache % 8 == 0 && kv.page % 4 == 0;
  static_assert(BM % 64 == 0 && BM <= THREADS, "whole wavefronts hold the rows' places");
  if (OUTMODE == 0 && kv.cache && t < BM) {
    slots[t] = slot;
    int way = vwide && kv_all_runs(slot, lane) ? KV_WAY_RUNS : 0;
    if (vwide && M >= KV_WALK_MIN_ROWS) {
      const int offset = kv_run_offset(slot, lane);
      way = way ? way : offset;
    }
    if (fr == 0) ways[t / 32] = way;
  }

#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int nl = wn + j * 32 + fr;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int ml = wm + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + (r % 4);
        if (OUTMODE == 0) ((bf16_t*)smem)[ml * LDT + nl] = f32_to_bf16(apply_act_bf16(acc[i][j][r] + bias[j], ACT));
        else ((float*)smem)[ml * LDT + nl] = apply_act(acc[i][j][r] + bias[j], ACT);
      }
  }
  lds_barrier();

  uint4 val[NCHK];
  int mm[NCHK], nn[NCHK];
#pragma unroll
  for (int k = 0; k < NCHK; ++k) {
    const int q = t + THREADS * k, row = q / CPR, c = q % CPR;
    mm[k] = m0 + row;
    nn[k] = n0 + c * CH;
    val[k] = *(const uint4*)(smem + (size_t)(row * LDT + c * CH) * ES);
  }
  const bool wide = (uintptr_t)ep.out % 16 == 0 && ep.ldo % CH == 0;
  if (wide) {
    if (OUTMODE == 2) {
      uint4 old[NCHK];
#pragma unroll
      for (int k = 0; k < NCHK; ++k) {
        const bool whole = mm[k] < M && nn[k] + CH <= N;
        old[k] = *(const uint4*)(whole ? (const void*)((const float*)ep.out + (size_t)mm[k] * ep.ldo + nn[k]) : safe);
      }
#pragma unroll
      for (int k = 0; k < NCHK; ++k) {
        const bool whole = mm[k] < M && nn[k] + CH <= N;     // (a select: what came from the safe place is dropped)
        val[k].x = whole ? __float_as_uint(__uint_as_float(old[k].x) + __uint_as_float(val[k].x)) : val[k].x;
        val[k].y = whole ? __float_as_uint(__uint_as_float(old[k].y) + __uint_as_float(val[k].y)) : val[k].y;
        val[k].z = whole ? __float_as_uint(__uint_as_float(old[k].z) + __uint_as_float(val[k].z)) : val[k].z;
        val[k].w = whole ? __float_as_uint(__uint_as_float(old[k].w) + __uint_as_float(val[k].w)) : val[k].w;
      }
    }
#pragma unroll
    for (int k = 0; k < NCHK; ++k)
      if (mm[k] < M && nn[k] + CH <= N) *(uint4*)((char*)ep.out + ((size_t)mm[k] * ep.ldo + nn[k]) * ES) = val[k];
  }
  // pieces that N cuts, and everything where the output's rows are not 16-byte aligned: by elements
  // (for +=, a piece that N cuts still holds the bare products here: only whole pieces were added to above)
#pragma unroll
  for (int k = 0; k < NCHK; ++k) {
    if (mm[k] >= M || nn[k] >= N || (wide && nn[k] + CH <= N)) continue;
    const uint32_t words[4] = {val[k].x, val[k].y, val[k].z, val[k].w};
#pragma unroll
    for (int e = 0; e < CH; ++e) {
      if (nn[k] + e >= N) continue;
      const size_t o = (size_t)mm[k] * ep.ldo + nn[k] + e;
      if (OUTMODE == 0) ((bf16_t*)ep.out)[o] = (bf16_t)(words[e / 2] >> (16 * (e % 2)));
      else if (OUTMODE == 1) ((float*)ep.out)[o] = __uint_as_float(words[e % 4]);
      else ((float*)ep.out)[o] += __uint_as_float(words[e % 4]);
    }
  }

  // A fused q|k|v projection: the k and v columns also go to the rows' places in the paged cache.
  // Keys are rows there: a piece of 8 columns is a piece of the key's row.  Values are dimension-major
  // (dimension d of a page's rows side by side): 4 consecutive tile rows of one column are one 8-byte
  // piece where their places are 4 consecutive rows of one page from a multiple of 4 on (a prompt
  // portion mostly is), and go entry by entry otherwise.
  if (OUTMODE == 0 && kv.cache) {
    // (the page size is a power of two, checked on the host: a place splits into page and row by shift and mask)
    const int lgp = 31 - __builtin_clz(kv.page), pmask = kv.page - 1;
    const bool kwide = (uintptr_t)kv.cache % 16 == 0 && kv.D % 8 == 0 && kv.q_cols % 8 == 0;
    const int v0 = kv.q_cols + kv.kv_cols;                              // the first value column
#pragma unroll
    for (int k = 0; k < NCHK; ++k) {
      const int slot = slots[mm[k] - m0];
      if (slot < 0 || nn[k] >= N || nn[k] + 8 <= kv.q_cols || nn[k] >= v0) continue;
      const int pg = slot >> lgp, prow = slot & pmask;
      if (kwide) {                              // eight dimensions of one key: one piece of its row
        const int c2 = nn[k] - kv.q_cols, h = c2 / kv.D, d = c2 % kv.D;
        *(uint4*)((bf16_t*)kv.cache + cache_k_row(pg, h, prow, kv.Hkv, kv.page, kv.D) + d) = val[k];
        continue;
      }
      const uint32_t words[4] = {val[k].x, val[k].y, val[k].z, val[k].w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (nn[k] + e >= kv.q_cols && nn[k] + e < v0)
          kv_scatter_bits(kv, pg, prow, nn[k] + e, (bf16_t)(words[e / 2] >> (16 * (e % 2))));
    }
    // Values: straight from the accumulators (a lane holds 4 consecutive rows of its column, r % 4; the lane of the other
    // half holds the 4 rows beside them), or from the parked tile, a column a lane; see kv_all_runs.
    const long long page_stride = 2LL * kv.Hkv * kv.page * kv.D;
    bf16_t* vb = (bf16_t*)kv.cache;
    if (n0 + wn + BN / WN <= v0 || n0 + wn >= N) return;                // (no value column among the wavefront's)
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int way = __builtin_amdgcn_readfirstlane(ways[wm / 32 + i]);
      if (__builtin_expect(way == KV_WAY_RUNS, 1)) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = n0 + wn + j * 32 + fr;
          if (n < v0 || n >= N) continue;
          const int cc = n - v0;
          const int vcol = (kv.Hkv + cc / kv.D) * kv.page * kv.D + (cc % kv.D) * kv.page;   // the column's run in a page
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            uint32_t w2[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
              w2[e] = pack2_bf16(apply_act_bf16(acc[i][j][4 * q + 2 * e] + bias[j], ACT),
                                 apply_act_bf16(acc[i][j][4 * q + 2 * e + 1] + bias[j], ACT));
            const int s0 = slots[wm + i * 32 + 8 * q + 4 * (lane / 32)];
            *(uint2*)(vb + vcol + (long long)(s0 >> lgp) * page_stride + (s0 & pmask)) = make_uint2(w2[0], w2[1]);
          }
        }
        continue;
      }
      if (way == 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = n0 + wn + j * 32 + fr;
          if (n < v0 || n >= N) continue;
          const int cc = n - v0;
          const int vcol = (kv.Hkv + cc / kv.D) * kv.page * kv.D + (cc % kv.D) * kv.page;   // the column's run in a page
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            uint32_t w2[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
              w2[e] = pack2_bf16(apply_act_bf16(acc[i][j][4 * q + 2 * e] + bias[j], ACT),
                                 apply_act_bf16(acc[i][j][4 * q + 2 * e + 1] + bias[j], ACT));
            kv_store_run(vb + vcol, *(const uint4*)&slots[wm + i * 32 + 8 * q + 4 * (lane / 32)], make_uint2(w2[0], w2[1]), vwide, page_stride, lgp, pmask);
          }
        }
        continue;
      }
      static_assert(BN / WN <= 64, "a column a lane");
      const int n = n0 + wn + lane, cc = n - v0;
      const bool mine = lane < BN / WN && cc >= 0 && n < N;
      bf16_t* const dst = mine ? vb + (long long)(kv.Hkv + cc / kv.D) * kv.page * kv.D + (cc % kv.D) * kv.page : nullptr;
      kv_store_values32<LDT>((const bf16_t*)smem + (wm + i * 32) * LDT + wn + lane % (BN / WN),
                             slots[wm + i * 32 + lane % 32], way, dst, page_stride, lgp, pmask);
    }
  }
}

// Grouped products: the rows of a come in groups of `rows` (a multiple of the tile's rows), and group i is
// multiplied with the matrix w + tile_group[i] * stride (a stack of matrices of one shape: the experts of a
// feed-forward); a group whose entry is negative is not used and its tiles leave at once.  No grouping: null.
struct Grouping {
  const int* tile_group;
  long stride;
  int rows;
};

template <int BM, int BN, int WM, int WN, int PF_SLABS, int ACT, int OUTMODE, bool KTAIL>
__device__ __forceinline__ void
gemm_tile_body(const bf16_t* __restrict__ a, int lda, const bf16_t* __restrict__ w, int ldw,
               const Epilogue& ep, const KvScatter& kv, int M, int N, int K, int tiles_m, int tiles_n,
               char* smem, const Grouping& gr, bool grouped) {
  bf16_t (*As)[BM * LDS_LD] = (bf16_t (*)[BM * LDS_LD])smem;
  bf16_t (*Ws)[BN * LDS_LD] = (bf16_t (*)[BN * LDS_LD])(smem + 2 * BM * LDS_LD * sizeof(bf16_t));
  constexpr int THREADS = WM * WN * 64;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;       // MFMA tiles per wavefront
  constexpr int CA = BM * 8 / THREADS, CW = BN * 8 / THREADS; // 16-byte chunks per thread and slab
  static_assert(BM * 8 % THREADS == 0 && BN * 8 % THREADS == 0, "tile does not split over the threads");
  static_assert(PF_SLABS == 2 || PF_SLABS == 4, "two or four slabs in flight");

  // Blocks that follow each other in launch order land on different XCDs (8 of them, each with
  // its own L2).  Give each XCD a contiguous run of tiles, m fastest, so that the blocks of one
  // XCD share slabs of w.
  const int nblocks = tiles_m * tiles_n;
  int pid = blockIdx.x;
  {
    const int per = nblocks / 8, rem = nblocks % 8;
    const int xcd = pid % 8, local = pid / 8;
    pid = xcd * per + (xcd < rem ? xcd : rem) + local;
  }
  const int tm = pid % tiles_m, tn = pid / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;
  if (grouped) {                            // (the same for the whole workgroup, before any barrier)
    const int g = gr.tile_group[m0 / gr.rows];
    if (g < 0) return;
    w += (size_t)g * gr.stride;
  }

  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // Loads are never conditional (a conditional load becomes a branch that serialises the slab's
  // loads).  Rows past the edge of a or w read the last row instead: what they produce is never
  // stored.  Chunks past K (KTAIL: K is no multiple of the slab) read the row's first chunk and are
  // replaced by zero afterwards; that replacement makes the compiler wait for loads early, so it is
  // compiled only where it is needed.  (The row's first chunk, not this thread's chunk of slab 0:
  // with K < 64 that one lies past K too, in the next row or, for the last row, past the tensor.)  PF_SLABS slabs are in flight in registers at any time: one slab's
  // products take far less time than a load, so the distance between asking and needing is what
  // keeps the matrix cores fed.
  uint4 ra[PF_SLABS][CA], rw[PF_SLABS][CW];
  const uint4 zero = make_uint4(0, 0, 0, 0);
  const bf16_t* pa[CA];
  const bf16_t* pw[CW];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int c = t + THREADS * i, row = m0 + c / 8;
    pa[i] = a + (size_t)(row < M ? row : M - 1) * lda + (c % 8) * 8;
  }
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int c = t + THREADS * i, row = n0 + c / 8;
    pw[i] = w + (size_t)(row < N ? row : N - 1) * ldw + (c % 8) * 8;
  }
  const int kc_t = (t % 8) * 8;                     // this thread's chunk offset inside a slab (THREADS % 8 == 0)
#define TILE_FETCH(stage, k0)                                   \
  {                                                             \
    const bool kin = !KTAIL || (k0) + kc_t < K;                 \
    const int ks = kin ? (k0) : -kc_t;                          \
    _Pragma("unroll") for (int i = 0; i < CA; ++i) {            \
      ra[stage][i] = load16(pa[i] + ks);                        \
      if (KTAIL && !kin) ra[stage][i] = zero;                   \
    }                                                           \
    _Pragma("unroll") for (int i = 0; i < CW; ++i) {            \
      rw[stage][i] = load16(pw[i] + ks);                        \
      if (KTAIL && !kin) rw[stage][i] = zero;                   \
    }                                                           \
  }
#define TILE_STASH(stage, buf)                                              \
  {                                                                         \
    _Pragma("unroll") for (int i = 0; i < CA; ++i) {                        \
      const int c = t + THREADS * i, row = c / 8, kc = (c % 8) * 8;         \
      *(uint4*)&As[buf][row * LDS_LD + kc] = ra[stage][i];                  \
    }                                                                       \
    _Pragma("unroll") for (int i = 0; i < CW; ++i) {                        \
      const int c = t + THREADS * i, row = c / 8, kc = (c % 8) * 8;         \
      *(uint4*)&Ws[buf][row * LDS_LD + kc] = rw[stage][i];                  \
    }                                                                       \
  }
  const int fr = lane % 32, fk = (lane / 32) * 8;
  const int nslab = (K + BKT - 1) / BKT;
#pragma unroll
  for (int j = 0; j < PF_SLABS; ++j)
    if (j < nslab) TILE_FETCH(j, j * BKT);
  // The bias is asked for behind the first slabs, as raw bits from a place that always exists, and has long arrived when
  // the products are done: a load inside the epilogue's conditions would make every store after it
  // wait for the one before.
  const bool bias_bf16 = ep.bias_dtype == DA_BF16;
  uint32_t braw[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 32 + fr;
    const bool has = ep.bias && n < N;
    const void* src = has ? ep.bias : (const void*)w;
    const int idx = has ? n : 0;
    braw[j] = bias_bf16 ? (uint32_t)((const bf16_t*)src)[idx] : ((const uint32_t*)src)[idx];
  }
  // ... and so is the place in the cache of the tile row that this thread puts into LDS
  int slot = -1;
  if (OUTMODE == 0) {
    const bool has = kv.cache && t < BM && m0 + t < M;
    const int place = *(has ? kv.slot_map + m0 + t : (const int*)w);
    slot = has ? place : -1;
  }
  // (the arguments that only the epilogue uses, too: a line of them asked for there would be waited for there)
  da_read_arg(ep.out);
  da_read_arg(ep.ldo);
  if (OUTMODE == 0) {
    da_read_arg(kv.q_cols);
    da_read_arg(kv.Hkv);
    da_read_arg(kv.page);
  }
  TILE_STASH(0, 0);
  lds_barrier();
  // One slab: stage j's registers went to LDS before the last barrier and take the slab PF_SLABS
  // further on; the products of slab sidx come out of LDS buffer j & 1 (= sidx & 1, PF_SLABS is
  // even); the next slab's registers go to the other buffer, which was last read before the
  // previous barrier.
#define TILE_STEP(j, sidx, want_fetch, want_stash)                                                              \
  {                                                                                                             \
    constexpr int buf = (j) & 1;                                                                                \
    if (want_fetch) TILE_FETCH(j, ((sidx) + PF_SLABS) * BKT);                                                   \
    _Pragma("unroll") for (int kk = 0; kk < BKT; kk += 16) {                                                    \
      bf16x8_t af[TM], bf[TN];                                                                                  \
      _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                            \
        af[i] = __builtin_bit_cast(bf16x8_t, *(const uint4*)&As[buf][(wm + i * 32 + fr) * LDS_LD + kk + fk]);   \
      _Pragma("unroll") for (int jj = 0; jj < TN; ++jj)                                                         \
        bf[jj] = __builtin_bit_cast(bf16x8_t, *(const uint4*)&Ws[buf][(wn + jj * 32 + fr) * LDS_LD + kk + fk]); \
      _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                            \
        _Pragma("unroll") for (int jj = 0; jj < TN; ++jj)                                                       \
          acc[i][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[jj], acc[i][jj], 0, 0, 0);             \
    }                                                                                                           \
    if (want_stash) TILE_STASH(((j) + 1) % PF_SLABS, buf ^ 1);                                                  \
    lds_barrier();                                                                                              \
  }
  // The steady state has no branches, so that the compiler counts the loads in flight exactly and
  // waits for the oldest slab only; the last slabs run through the same steps with conditions.
  int base = 0;
  for (; base + 2 * PF_SLABS <= nslab; base += PF_SLABS) {
    TILE_STEP(0, base, true, true);
    TILE_STEP(1, base + 1, true, true);
    if constexpr (PF_SLABS == 4) {
      TILE_STEP(2, base + 2, true, true);
      TILE_STEP(3, base + 3, true, true);
    }
  }
  for (; base < nslab; base += PF_SLABS) {
    if (base < nslab) TILE_STEP(0, base, base + PF_SLABS < nslab, base + 1 < nslab);
    if (base + 1 < nslab) TILE_STEP(1, base + 1, base + 1 + PF_SLABS < nslab, base + 2 < nslab);
    if constexpr (PF_SLABS == 4) {
      if (base + 2 < nslab) TILE_STEP(2, base + 2, base + 2 + PF_SLABS < nslab, base + 3 < nslab);
      if (base + 3 < nslab) TILE_STEP(3, base + 3, base + 3 + PF_SLABS < nslab, base + 4 < nslab);
    }
  }
#undef TILE_STEP
#undef TILE_FETCH
#undef TILE_STASH

  float bias[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) bias[j] = !ep.bias ? 0.f : (bias_bf16 ? __uint_as_float(braw[j] << 16) : __uint_as_float(braw[j]));
  tile_epilogue<BM, BN, WM, WN, ACT, OUTMODE>(acc, bias, smem, (const void*)w, ep, kv, slot, M, N, m0, n0);
}

template <int BM, int BN, int WM, int WN, int PF, int ACT, int OUTMODE>
__global__ void __launch_bounds__(WM * WN * 64)
gemm_tile_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const void* bias, int lda, int ldw, int M, int N, int K, int tiles_m,
                 int tiles_n, int flags, void* out, int ldo, KvScatter kv, Grouping gr) {
  // (the first 14 words are in registers when the wavefront starts; `flags`: the bias's type, and 0x100 where the rows are grouped)
  const Epilogue ep{bias, flags & 0xff, ACT, OUTMODE == 2, out, OUTMODE == 0 ? DA_BF16 : DA_F32, ldo};
  const bool grouped = flags & 0x100;
  // two buffers of a slab of a and of w; the epilogue parks the tile's results in the same memory
  constexpr int SLAB_BYTES = 2 * (BM + BN) * LDS_LD * (int)sizeof(bf16_t);
  constexpr int OUT_BYTES = tile_out_bytes<BM, BN, OUTMODE>() + tile_slot_bytes<BM, OUTMODE>();
  __shared__ __attribute__((aligned(16))) char smem[SLAB_BYTES > OUT_BYTES ? SLAB_BYTES : OUT_BYTES];      // shared by the two bodies
  if (K % BKT == 0) gemm_tile_body<BM, BN, WM, WN, PF, ACT, OUTMODE, false>(a, lda, w, ldw, ep, kv, M, N, K, tiles_m, tiles_n, smem, gr, grouped);
  else gemm_tile_body<BM, BN, WM, WN, PF, ACT, OUTMODE, true>(a, lda, w, ldw, ep, kv, M, N, K, tiles_m, tiles_n, smem, gr, grouped);
}

template <int BM, int BN, int WM, int WN, int PF, int ACT>
static void launch_tile_act(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep,
                            const KvScatter& kv, int M, int N, int K, const Grouping& gr) {
  const int tiles_m = da_ceil_div(M, BM), tiles_n = da_ceil_div(N, BN);
  const dim3 grid(tiles_m * tiles_n), block(WM * WN * 64);
  const int flags = ep.bias_dtype | (gr.tile_group ? 0x100 : 0);
  if (ep.accumulate)
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, PF, ACT, 2>), grid, block, 0, s, A, W, ep.bias, lda, ldw, M, N, K, tiles_m, tiles_n, flags, ep.out, ep.ldo, kv, gr);
  else if (ep.out_dtype == DA_F32)
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, PF, ACT, 1>), grid, block, 0, s, A, W, ep.bias, lda, ldw, M, N, K, tiles_m, tiles_n, flags, ep.out, ep.ldo, kv, gr);
  else
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, PF, ACT, 0>), grid, block, 0, s, A, W, ep.bias, lda, ldw, M, N, K, tiles_m, tiles_n, flags, ep.out, ep.ldo, kv, gr);
}

template <int BM, int BN, int WM, int WN, int PF>
static void launch_tile(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep,
                        const KvScatter& kv, int M, int N, int K, const Grouping& gr = Grouping{nullptr, 0, 0}) {
  switch (ep.act) {
    case DA_ACT_GELU_TANH: launch_tile_act<BM, BN, WM, WN, PF, DA_ACT_GELU_TANH>(s, A, lda, W, ldw, ep, kv, M, N, K, gr); break;
    case DA_ACT_GELU_ERF: launch_tile_act<BM, BN, WM, WN, PF, DA_ACT_GELU_ERF>(s, A, lda, W, ldw, ep, kv, M, N, K, gr); break;
    case DA_ACT_RELU: launch_tile_act<BM, BN, WM, WN, PF, DA_ACT_RELU>(s, A, lda, W, ldw, ep, kv, M, N, K, gr); break;
    case DA_ACT_SILU: launch_tile_act<BM, BN, WM, WN, PF, DA_ACT_SILU>(s, A, lda, W, ldw, ep, kv, M, N, K, gr); break;
    case DA_ACT_RELU2: launch_tile_act<BM, BN, WM, WN, PF, DA_ACT_RELU2>(s, A, lda, W, ldw, ep, kv, M, N, K, gr); break;
    default: launch_tile_act<BM, BN, WM, WN, PF, DA_ACT_NONE>(s, A, lda, W, ldw, ep, kv, M, N, K, gr); break;
  }
}

// ---------------------------------------------------------------------------------------------
// M <= 64.  A workgroup owns 16 output columns and MT row tiles of 16 (all of them, or with few
// columns some: blockIdx.y); wavefront v of NW takes the steps v, v+NW, ... of 64 elements of k, so
// that NW chains of loads run side by side; MFMA 16x16x32; the wavefronts' sums are added through
// LDS in a fixed order.  The operands come in whole cache lines: a load takes 8 rows x 128 bytes,
// the wavefront parks a step in its own piece of LDS and reads the fragments from there.  (Loaded
// straight in fragment order, 16 rows x 64 bytes a load, they pass a compute unit's L1 at a third
// of the rate, and that rate, not the memory's, bounds a workgroup.)
// ---------------------------------------------------------------------------------------------
// AL: loads of 8 rows that cover the workgroup's rows of a (1: up to 8 rows; else two a row tile);
// COLS: 16 output columns a workgroup, or 8 (the fragment of w then holds them twice and half of the
// result is dropped: with few columns twice the workgroups pull on memory).
// GATED: w is [2 N, K], gate rows and then up rows; a workgroup's 16 columns are 8 gate columns and the same 8 up columns, and what leaves
// is gated_mid of their 32-bit sums in bfloat16 (da_gemm_bf16_gated; `gate_limit` is its).
template <int AL, int COLS, int NW, int UNROLL, bool GATED = false>
__global__ void __launch_bounds__(NW * 64)
gemm_skinny_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const void* bias, void* out, int lda, int ldw, int ldo,
                   int M, int N, int K, EpilogueRest er, KvScatter kv, float gate_limit) {
  static_assert(!GATED || COLS == 16, "eight columns of each");
  constexpr int MT = (AL + 1) / 2, WL = COLS / 8;    // row tiles of 16; loads of 8 rows that cover w's columns
  constexpr int AR = MT * 16, TR = AR + COLS;        // rows of a; rows of a step: a's, then w's
  static_assert(COLS == 8 || COLS == 16, "8 or 16 columns a workgroup");
  // The wavefronts' partial sums lie behind the parked steps, where that leaves room for the workgroups that registers allow; else they
  // take their place once all products are done, behind a barrier more.
  constexpr int STAGE_BYTES = NW * TR * SK_LD * 2, RED_BYTES = NW * AR * (COLS + 1) * 4;
  constexpr bool APART = STAGE_BYTES + RED_BYTES <= (NW == 4 ? 32 : 80) * 1024;
  __shared__ __attribute__((aligned(16))) char smem[APART ? STAGE_BYTES + RED_BYTES : (STAGE_BYTES > RED_BYTES ? STAGE_BYTES : RED_BYTES)];
  bf16_t (*stage)[TR * SK_LD] = (bf16_t (*)[TR * SK_LD])smem;
  float (*red)[AR][COLS + 1] = (float (*)[AR][COLS + 1])(smem + (APART ? STAGE_BYTES : 0));
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int n0 = blockIdx.x * (GATED ? 8 : COLS);
  const int r0 = blockIdx.y * AR;                    // the workgroup's first row
  const int lr = lane / 8, lc = (lane % 8) * 8;      // a load: row lr of 8, 16-byte piece lane % 8
  const int fr = lane % 16, fk = (lane / 16) * 8;    // a fragment: row fr of 16, k-group lane / 16
  const bf16_t* pa[AL];
  const bf16_t* pw[WL];
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    const int m = r0 + i * 8 + lr;
    pa[i] = a + (size_t)(m < M ? m : 0) * lda + lc;
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int n = n0 + (GATED ? 0 : i * 8) + lr;
    pw[i] = w + (size_t)((n < N ? n : 0) + (GATED ? i * N : 0)) * ldw + lc;
  }
  // What the epilogue needs is asked for behind the last group of operands, as raw bits from places that always exist: its arguments
  // lie in other lines than the operands' and are still on the way when those are asked for.
  constexpr int OC = GATED ? 8 : COLS;               // columns that leave
  constexpr int EPT = (AR * OC + NW * 64 - 1) / (NW * 64);
  uint32_t e_braw[EPT];
  float e_old[EPT];
  int e_slot[EPT];
  KvColumn e_col[EPT];
  auto load_epilogue = [&]() {
    da_read_arg(er.act);
    if constexpr (GATED) {
      da_read_arg(gate_limit);
      return;
    }
    da_read_arg(er.out_dtype);
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = t + j * NW * 64, m = r0 + e / COLS, n = n0 + e % COLS;
      const bool ok = e < AR * COLS && m < M && n < N;
      const void* bsrc = (ok && bias) ? bias : (const void*)w;
      const int bidx = (ok && bias) ? n : 0;
      e_braw[j] = er.bias_dtype == DA_BF16 ? (uint32_t)((const bf16_t*)bsrc)[bidx] : ((const uint32_t*)bsrc)[bidx];
      e_old[j] = *((ok && er.accumulate) ? (const float*)out + (size_t)m * ldo + n : (const float*)w);
      e_slot[j] = *((ok && kv.cache) ? kv.slot_map + m : (const int*)w);
      if (kv.cache) e_col[j] = kv_column(kv, n);
    }
  };
  floatx4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16_t* mine = stage[wave];
  // (With AL == 1 the rows 8..15 of the tile are never parked: whatever LDS holds there gives rows of
  // the result that are never stored.)
  // The wavefront's steps (v, v+NW, ...) go two at a time: all loads of both first, then each is
  // parked in LDS and multiplied.  The very last step may be the one that K cuts: lanes past K read
  // the row's first piece instead and park zeros.
  const int steps = (K + 63) / 64;
  int count = wave < steps ? (steps - wave + NW - 1) / NW : 0;
  int k0 = wave * 64;
  auto group = [&](auto gc, auto lastc) {
    constexpr int G = decltype(gc)::value;
    constexpr bool LAST = decltype(lastc)::value;
    uint4 av[G][AL], wv[G][WL];
    bool kin = true;
#pragma unroll
    for (int u = 0; u < G; ++u) {
      int kk = k0 + u * NW * 64;
      if (LAST && u == G - 1) {
        kin = kk + lc < K;
        kk = kin ? kk : -lc;
      }
#pragma unroll
      for (int i = 0; i < AL; ++i) av[u][i] = load16(pa[i] + kk);
#pragma unroll
      for (int i = 0; i < WL; ++i) wv[u][i] = load16(pw[i] + kk);
    }
    if (LAST) load_epilogue();
#pragma unroll
    for (int u = 0; u < G; ++u) {
#pragma unroll
      for (int i = 0; i < AL; ++i) *(uint4*)&mine[(i * 8 + lr) * SK_LD + lc] = av[u][i];
#pragma unroll
      for (int i = 0; i < WL; ++i) *(uint4*)&mine[(AR + i * 8 + lr) * SK_LD + lc] = wv[u][i];
      if (LAST && u == G - 1 && !kin) {        // past K: zeros over what the lane just parked
        const uint4 zero = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < AL; ++i) *(uint4*)&mine[(i * 8 + lr) * SK_LD + lc] = zero;
#pragma unroll
        for (int i = 0; i < WL; ++i) *(uint4*)&mine[(AR + i * 8 + lr) * SK_LD + lc] = zero;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
      for (int c = 0; c < 64; c += 32) {
        const bf16x8_t wf = __builtin_bit_cast(bf16x8_t, *(const uint4*)&mine[(AR + fr % COLS) * SK_LD + c + fk]);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const bf16x8_t af = __builtin_bit_cast(bf16x8_t, *(const uint4*)&mine[(i * 16 + fr) * SK_LD + c + fk]);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf, acc[i], 0, 0, 0);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    }
    k0 += G * NW * 64;
    count -= G;
  };
  while (count > UNROLL) group(std::integral_constant<int, UNROLL>{}, std::false_type{});
  switch (count) {
    case 4: if (UNROLL >= 4) group(std::integral_constant<int, (UNROLL >= 4 ? 4 : 1)>{}, std::true_type{}); break;
    case 3: if (UNROLL >= 3) group(std::integral_constant<int, (UNROLL >= 3 ? 3 : 1)>{}, std::true_type{}); break;
    case 2: if (UNROLL >= 2) group(std::integral_constant<int, (UNROLL >= 2 ? 2 : 1)>{}, std::true_type{}); break;
    case 1: group(std::integral_constant<int, 1>{}, std::true_type{}); break;
    default: load_epilogue(); break;
  }
  if (!APART) lds_barrier();
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (COLS == 16 || fr < COLS) red[wave][i * 16 + 4 * (lane / 16) + r][fr] = acc[i][r];
  lds_barrier();
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = t + j * NW * 64, ml = e / OC, m = r0 + ml, c = e % OC, n = n0 + c;
    if (e < AR * OC && m < M && n < N) {
      float v = red[0][ml][c];
#pragma unroll
      for (int v2 = 1; v2 < NW; ++v2) v += red[v2][ml][c];
      if constexpr (GATED) {
        float u = red[0][ml][8 + c];
#pragma unroll
        for (int v2 = 1; v2 < NW; ++v2) u += red[v2][ml][8 + c];
        ((bf16_t*)out)[(size_t)m * ldo + n] = f32_to_bf16(gated_mid<true>(v, u, er.act, gate_limit));
        continue;
      }
      const float e_bias = !bias ? 0.f : (er.bias_dtype == DA_BF16 ? __uint_as_float(e_braw[j] << 16) : __uint_as_float(e_braw[j]));
      v = er.out_dtype == DA_BF16 ? apply_act_bf16(v + e_bias, er.act) : apply_act(v + e_bias, er.act);
      const size_t o = (size_t)m * ldo + n;
      if (er.accumulate) ((float*)out)[o] = e_old[j] + v;
      else if (er.out_dtype == DA_BF16) ((bf16_t*)out)[o] = f32_to_bf16(v);
      else ((float*)out)[o] = v;
      if (kv.cache) kv_column_store(kv, e_col[j], e_slot[j], v);
    }
  }
}

// Whether a product of few rows goes to gemm_skinny32: more than 4,096 columns (fewer give no compute unit two workgroups of
// 16) and up to 8,192.  More than 16 rows: always (K from 64 to 8,192: 0.55 to 0.98 of the time of 16 columns a
// workgroup).  Up to 16 rows the rows are few bytes and two workgroups a compute unit hide more latency than one, so it
// pays only where the busiest compute unit pulls much less of w: with a long K and well below 32 columns a unit.
// Measured with cold weights, 16 columns against one workgroup a unit, both with 8 wavefronts:
//    8 rows: K = 1,600, N = 4,800 6.3 against 6.1 us, 8,192 7.0 / 7.8; K = 4,096, N = 4,112 10.6 / 9.2, 6,400 11.9 / 12.1, 8,192 13.1 / 16.3; K = 8,192, N = 6,400 23.8 / 21.7
//   16 rows: K = 1,600, N = 4,800 7.1 against 6.4 us, 5,888 6.9 / 6.7, 7,168 7.0 / 7.2; K = 3,072, N = 7,168 11.8 / 10.8, 7,680 11.9 / 11.2
// Its offsets of 64 rows are 32-bit: rows that lie further apart than 2^24 entries stay with 16 columns (the same bits).
static bool sk_one_a_unit(int M, int N, int K, int lda, int ldw) {
  const int cols = da_ceil_div(N, 256);              // of the busiest compute unit, where 16 a workgroup give it 32
  if (cols <= 16 || cols > 32 || lda > (1 << 24) || ldw > (1 << 24)) return false;
  if (M > 16) return true;
  if (M > 8) return (K >= 1280 && cols <= 23) || (K >= 3072 && cols <= 28);
  return (M > 4 && K >= 1280 && cols <= 20) || (K >= 3072 && cols <= 22 + K / 2048);
}

// The wavefronts that split K of a product of few rows, by K and N alone, so that a row's sums keep their order:
// 4 where the workgroups are many (a vocabulary: several then share a compute unit), else 8, or 12 for a long K where no compute
// unit has two workgroups (between 4,097 and 8,192 columns, K from 2,048 on, up to 16 rows 8 take 0.84 to 0.96 of 12's time).
static int sk_wavefronts(int N, int K) { return da_ceil_div(N, 16) > 1024 ? 4 : (K >= 2048 && (N <= 16 * 256 || N > 32 * 256) ? 12 : 8); }
// few columns and one row tile: 8 columns a workgroup
static bool sk_eight_columns(int M, int N, int nw) { return M <= 16 && nw != 4 && da_ceil_div(N, 16) < 128; }

template <int NW>
static int launch_skinny(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw,
                         const Epilogue& ep, const KvScatter& kv, int M, int N, int K) {
  const dim3 block(NW * 64);
  int mt = da_ceil_div(M, 16);
#define DA_SK_GO(AL, COLS, U) hipLaunchKernelGGL((gemm_skinny_kernel<AL, COLS, NW, U>), grid, block, 0, s, A, W, ep.bias, ep.out, lda, ldw, ep.ldo, M, N, K, epilogue_rest(ep), kv, 0.f)
  if (sk_eight_columns(M, N, NW)) {
    const dim3 grid(da_ceil_div(N, 8));
    if (M <= 8) DA_SK_GO(1, 8, 4); else DA_SK_GO(2, 8, 4);
    return 0;
  }
  if (NW == 8 && sk_one_a_unit(M, N, K, lda, ldw)) {
    const int cols = da_ceil_div(N, 256);            // every compute unit one workgroup
    const dim3 grid(da_ceil_div(N, cols));
#define DA_SK32_GO(AL, P) hipLaunchKernelGGL((gemm_skinny32_kernel<AL, 8, P, false>), grid, dim3(512), 0, s, A, W, ep.out, lda, ldw, ep.ldo, M, N, K, cols, K, ep.bias, epilogue_rest(ep), kv)
    // (steps in flight: what the registers of a workgroup that is alone on its compute unit allow)
    if (M <= 8) DA_SK32_GO(1, 4);
    else if (mt == 1) DA_SK32_GO(2, 4);
    else if (mt == 2) DA_SK32_GO(4, 3);
    else if (mt == 3) DA_SK32_GO(6, 2);
    else DA_SK32_GO(8, 2);
#undef DA_SK32_GO
    return 0;
  }
  dim3 grid(da_ceil_div(N, 16));
  // With few columns the row tiles are spread over more workgroups (blockIdx.y), as long as the chip
  // is not full: each then reads fewer rows of a.  A row's sums do not depend on it.
  for (int mb = 1; mb < mt; mb *= 2)
    if ((long)grid.x * da_ceil_div(mt, mb) <= 256) {
      grid.y = da_ceil_div(mt, mb);
      mt = mb;
      break;
    }
  DA_REQUIRE(mt >= 1 && mt <= 4, "gemm_bf16: %d row tiles", mt);
  // steps in flight: 16 to 20 loads of 16 bytes a lane
  if (mt == 1 && M <= 8) DA_SK_GO(1, 16, 4);
  else if (mt == 1) DA_SK_GO(2, 16, 4);
  else if (mt == 2) DA_SK_GO(4, 16, 3);
  else if (mt == 3) DA_SK_GO(6, 16, 2);
  else DA_SK_GO(8, 16, 2);
#undef DA_SK_GO
  return 0;
}

// ---------------------------------------------------------------------------------------------
// M <= 4, or 8 with a long K, and up to 2,048 columns (a decode step of a few requests).  MFMA 16x16x32 with pieces of k side by side: row 4 n + b
// of the left operand holds in k-group g the 8 elements from 8 (4 g + b) of a step of 128, of row n of 4 of w; column 4 m + b of
// the right operand the same of row m of 4 of a.  The result's entry (4 n + b, 4 m + b) is what the pieces b give, and four
// neighbouring lanes add up the four; the entries of unlike pieces are not looked at.  So four lanes that follow each other read 64
// consecutive bytes, which a compute unit takes at once; with a row a lane it takes them one at a time.  A workgroup owns
// 4 * NG columns; wavefront v of NW takes the steps v, v+NW, ...; the wavefronts' sums are added through LDS in a fixed order.
// ---------------------------------------------------------------------------------------------
template <int MG, int NG, int NW, int UNROLL>
__global__ void __launch_bounds__(NW * 64)
gemm_skinny4_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const void* bias, void* out, int lda, int ldw, int ldo,
                    int M, int N, int K, EpilogueRest er, KvScatter kv) {
  constexpr int ROWS = 4 * MG, COLS = NG * 4;
  __shared__ float red[NW][ROWS][COLS];
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int n0 = blockIdx.x * COLS;
  const int r4 = lane / 4 % 4, kb = (4 * (lane / 16) + lane % 4) * 8;
  const bf16_t* wp[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int n = n0 + g * 4 + r4;
    wp[g] = w + (size_t)(n < N ? n : 0) * ldw + kb;
  }
  const bf16_t* ap[MG];
#pragma unroll
  for (int i = 0; i < MG; ++i) ap[i] = a + (size_t)(4 * i + r4 < M ? 4 * i + r4 : 0) * lda + kb;
  // Four threads an output element: each sums a quarter of the wavefronts' sums, the first of them stores.  What the epilogue needs is
  // asked for behind the last operands, as in gemm_skinny.
  static_assert(NW % 4 == 0 && NW * 64 >= 4 * ROWS * COLS, "four threads an output element");
  const int e_id = t / 4, e_q = t % 4;
  const int e_m = e_id / COLS, e_c = e_id % COLS, e_n = n0 + e_c;
  const bool e_st = e_m < M && e_m < ROWS && e_n < N && e_q == 0;
  uint32_t e_braw;
  float e_old;
  int e_slot;
  KvColumn e_col;
  auto load_epilogue = [&]() {
    da_read_arg(er.act);
    da_read_arg(er.out_dtype);
    const void* e_bsrc = (e_st && bias) ? bias : (const void*)w;
    const int e_bidx = (e_st && bias) ? e_n : 0;
    e_braw = er.bias_dtype == DA_BF16 ? (uint32_t)((const bf16_t*)e_bsrc)[e_bidx] : ((const uint32_t*)e_bsrc)[e_bidx];
    e_old = *((e_st && er.accumulate) ? (const float*)out + (size_t)e_m * ldo + e_n : (const float*)w);
    e_slot = *((e_st && kv.cache) ? kv.slot_map + e_m : (const int*)w);
    if (kv.cache) e_col = kv_column(kv, e_n);
  };

  floatx4 acc[MG][NG];
#pragma unroll
  for (int i = 0; i < MG; ++i)
#pragma unroll
    for (int j = 0; j < NG; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  // The wavefront's steps go in groups of UNROLL and one last group of what is left: a group is
  // nothing but its loads, all in flight at once, and then its products.  The last step of the last
  // group may be the one that K cuts: lanes past K read the row's first piece instead and give
  // zeros for both (a multiple of 8 elements is in or out as a whole).
  const int steps = (K + 127) / 128;
  int count = wave < steps ? (steps - wave + NW - 1) / NW : 0;
  int k0 = wave * 128;
  auto group = [&](auto gc, auto lastc) {
    constexpr int G = decltype(gc)::value;
    constexpr bool LAST = decltype(lastc)::value;
    uint4 av[G][MG], wv[G][NG];
    bool kin = true;
#pragma unroll
    for (int u = 0; u < G; ++u) {
      int kk = k0 + u * NW * 128;
      if (LAST && u == G - 1) {
        kin = kk + kb < K;
        kk = kin ? kk : -kb;
      }
#pragma unroll
      for (int i = 0; i < MG; ++i) av[u][i] = load16(ap[i] + kk);
#pragma unroll
      for (int j = 0; j < NG; ++j) wv[u][j] = load16(wp[j] + kk);
    }
    if (LAST) load_epilogue();
    __builtin_amdgcn_sched_barrier(0);       // (else loads are pushed down among the products to save registers)
#pragma unroll
    for (int u = 0; u < G; ++u) {
      if (LAST && u == G - 1 && !kin) {
#pragma unroll
        for (int i = 0; i < MG; ++i) av[u][i] = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NG; ++j) wv[u][j] = make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < MG; ++i)
#pragma unroll
        for (int j = 0; j < NG; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wv[u][j]), __builtin_bit_cast(bf16x8_t, av[u][i]), acc[i][j], 0, 0, 0);
    }
    k0 += G * NW * 128;
    count -= G;
  };
  while (count > UNROLL) group(std::integral_constant<int, UNROLL>{}, std::false_type{});
  switch (count) {
    case 4: if (UNROLL >= 4) group(std::integral_constant<int, (UNROLL >= 4 ? 4 : 1)>{}, std::true_type{}); break;
    case 3: if (UNROLL >= 3) group(std::integral_constant<int, (UNROLL >= 3 ? 3 : 1)>{}, std::true_type{}); break;
    case 2: if (UNROLL >= 2) group(std::integral_constant<int, (UNROLL >= 2 ? 2 : 1)>{}, std::true_type{}); break;
    case 1: group(std::integral_constant<int, 1>{}, std::true_type{}); break;
    default: load_epilogue(); break;
  }
  // a lane has column 4 m + b and the rows 4 n .. 4 n + 3, n its quarter of the wavefront: of these, row 4 n + b
#pragma unroll
  for (int i = 0; i < MG; ++i)
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const float d01 = lane & 1 ? acc[i][j][1] : acc[i][j][0], d23 = lane & 1 ? acc[i][j][3] : acc[i][j][2];
      const float v = group_sum<4>(lane & 2 ? d23 : d01);
      if (lane % 4 == 0) red[wave][4 * i + r4][j * 4 + lane / 16] = v;
    }
  lds_barrier();
  if (e_m < ROWS) {                       // whole quads
    // thread e_q of the four takes the wavefronts e_q, e_q + 4, ...
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < NW / 4; ++i) v += red[e_q + 4 * i][e_m][e_c];
    v = group_sum<4>(v);
    if (e_st) {
      const float e_bias = !bias ? 0.f : (er.bias_dtype == DA_BF16 ? __uint_as_float(e_braw << 16) : __uint_as_float(e_braw));
      v = er.out_dtype == DA_BF16 ? apply_act_bf16(v + e_bias, er.act) : apply_act(v + e_bias, er.act);
      const size_t o = (size_t)e_m * ldo + e_n;
      if (er.accumulate) ((float*)out)[o] = e_old + v;
      else if (er.out_dtype == DA_BF16) ((bf16_t*)out)[o] = f32_to_bf16(v);
      else ((float*)out)[o] = v;
      if (kv.cache) kv_column_store(kv, e_col, e_slot, v);
    }
  }
}

// The wavefronts by K alone, so a row's sums keep their order; columns a workgroup so that the operands of a are no more than those of w
// where that pays.  us, cold weights, recorded one behind the other, 4x4x4 with a row a lane (up to 4 rows) or gemm_skinny (8 rows) -> this:
//   1 row   1,600 x 6,400 6.3 -> 5.7, 768 x 3,072 3.8 -> 3.2, 1,600 x 1,600 3.7 -> 3.4, 768 x 768 2.7 -> 2.6
//   4 rows  1,600 x 6,400 7.3 -> 6.1, 768 x 3,072 4.3 -> 3.5, 1,600 x 1,600 4.0 -> 3.6, 2,048 x 8,192 9.4 -> 7.8
//   8 rows  1,600 x 6,400 7.4 -> 7.1, 768 x 3,072 4.5 -> 4.0, 1,024 x 4,096 5.5 -> 4.4; 1,600 x 1,600 3.8 -> 3.9 (so from K = 2,048 on);
//           2,048 x 2,048 4.0 -> 4.2, 2,048 x 3,072 4.5 -> 4.7, 2,048 x 4,096 5.5 -> 5.5, but 1,984 x 2,048 level (so not where every compute unit has one of its
//           workgroups, up to K = 3,584)
// The weights alone, read and dropped, take 5.2, 2.5 and 2.6 us (1,600 x 6,400, 768 x 3,072, 1,600 x 1,600).
#define SK4_ROWS 4
#define SK4_LONG_ROWS 8
#define SK4_LONG_K 2048
#define SK4_COLS 2048
static bool sk4_takes(int M, int N, int K) {
  return N <= SK4_COLS && (M <= SK4_ROWS || (M <= SK4_LONG_ROWS && K >= SK4_LONG_K && (N <= 1984 || K >= 3584)));
}
// 1 when a product goes there
extern "C" int da_gemm_pieces_takes(int M, int N, int K) { return M > 0 && sk4_takes(M, N, K); }
static void launch_skinny4(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep, const KvScatter& kv, int M,
                           int N, int K) {
#define DA_SK4_GO(MG, NG, NW, U) hipLaunchKernelGGL((gemm_skinny4_kernel<MG, NG, NW, U>), dim3(da_ceil_div(N, 4 * NG)), dim3(NW * 64), 0, s, A, W, ep.bias, ep.out, lda, ldw, ep.ldo, M, N, K, epilogue_rest(ep), kv)
  if (M > SK4_ROWS) {                                     // (K from SK4_LONG_K on)
    if (N <= 1024) DA_SK4_GO(2, 1, 8, 4);
    else DA_SK4_GO(2, 2, 8, 3);
  } else if (K < 1024) DA_SK4_GO(1, 1, 4, 4);
  else if (N <= 1024 || K < 4096) DA_SK4_GO(1, 1, 8, 4);
  else DA_SK4_GO(1, 2, 8, 4);
#undef DA_SK4_GO
}

// 1 when a product of so many rows and columns goes to the kernels for few rows
extern "C" int da_gemm_few_rows(int M, int N) {
  return M <= 32 || (M <= 64 && N <= 8192);           // (a vocabulary with more than 32 rows: block tiles reuse the rows of a)
}

static int gemm_bf16_checks(const void* a, int lda, const void* w, int ldw, int act, int accumulate, int out_dtype, int ldo, int M,
                            int N, int K) {
  DA_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_bf16: bad sizes M=%d N=%d K=%d", M, N, K);
  DA_REQUIRE(K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0,
             "gemm_bf16: K, lda and ldw must be multiples of 8 (K=%d lda=%d ldw=%d)", K, lda, ldw);
  DA_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_bf16: operands must be 16-byte aligned");
  DA_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm_bf16: leading sizes too small");
  DA_REQUIRE(!accumulate || out_dtype == DA_F32, "gemm_bf16: accumulation needs a 32-bit output");
  DA_REQUIRE(act >= DA_ACT_NONE && act <= DA_ACT_LAST, "gemm_bf16: unknown activation %d", act);
  return 0;
}

static int gemm_bf16_launch(const void* a, int lda, const void* w, int ldw, const Epilogue& ep, const KvScatter& kv, int M, int N,
                            int K, void* stream);

// 1 where the gate and up products of few rows and their activation are one kernel: where the product of both matrices' columns would go to
// gemm_skinny with 16 columns a workgroup and all rows in it (or, 5 to 8 rows with a long K, to gemm_skinny4: K = 2,048, 2 x 1,024 columns the product
// alone 3.9, this 3.7).  One rounding to bfloat16 and one launch fewer; us, the product and the
// activation's kernel / this, cold weights: 8 rows, K = 1,024, 2 x 2,752 columns 6.7 / 4.5; K = 768, 2 x 2,048 columns 1 row 5.2 / 3.4, 64 rows
// 7.5 / 4.5; K = 3,072, 2 x 8,192 columns 8 rows 19.9 / 17.3.
extern "C" int da_gemm_gated_takes(int M, int inner, int K) {
  const long N = 2L * inner;
  if (M < 1 || inner < 1 || K < 8 || K % 8 || N > 16 * 1024 || !da_gemm_few_rows(M, (int)N) || (M <= SK4_ROWS && N <= SK4_COLS)) return 0;
  if (sk_eight_columns(M, (int)N, sk_wavefronts((int)N, K)) || (sk_wavefronts((int)N, K) == 8 && sk_one_a_unit(M, (int)N, K, K, K))) return 0;
  return M <= 16 || da_ceil_div(N, 16) >= 256;
}
// mid = act(a @ gate.T) * (a @ up.T), w the gate rows and then the up rows: [2 inner, K].
extern "C" int da_gemm_bf16_gated(const void* a, int lda, const void* w, int ldw, void* mid, int ldm, int M, int inner, int K, int act, float limit,
                                  void* stream) {
  if (gemm_bf16_checks(a, lda, w, ldw, act, 0, DA_BF16, ldm, M, inner, K)) return 1;
  DA_REQUIRE(act != DA_ACT_GLU_CAPPED || limit > 0.f, "gemm_bf16_gated: the capped form needs a positive limit");
  if (M == 0) return 0;
  DA_REQUIRE(da_gemm_gated_takes(M, inner, K), "gemm_bf16_gated: %d rows, 2 x %d columns, K=%d are not taken", M, inner, K);
  const dim3 grid(da_ceil_div(inner, 8));
  const int nw = sk_wavefronts(2 * inner, K);
#define DA_SKG_GO(AL, NW, U) hipLaunchKernelGGL((gemm_skinny_kernel<AL, 16, NW, U, true>), grid, dim3(NW * 64), 0, (hipStream_t)stream, (const bf16_t*)a, \
                                                (const bf16_t*)w, nullptr, mid, lda, ldw, ldm, M, inner, K, EpilogueRest{0, act, 0, DA_BF16}, KvScatter{}, limit)
#define DA_SKG_ROWS(NW)                          \
  do {                                           \
    if (M <= 8) DA_SKG_GO(1, NW, 4);             \
    else if (M <= 16) DA_SKG_GO(2, NW, 4);       \
    else if (M <= 32) DA_SKG_GO(4, NW, 3);       \
    else if (M <= 48) DA_SKG_GO(6, NW, 2);       \
    else DA_SKG_GO(8, NW, 2);                    \
  } while (0)
  if (nw == 12) DA_SKG_ROWS(12); else DA_SKG_ROWS(8);
#undef DA_SKG_ROWS
#undef DA_SKG_GO
  DA_CHECK_LAUNCH("gemm_bf16_gated");
  return 0;
}

extern "C" int da_gemm_bf16(const void* a, int lda, const void* w, int ldw, const void* bias, int bias_dtype,
                            int act, int accumulate, void* out, int out_dtype, int ldo, int M, int N, int K,
                            void* kv_cache, const int* slot_map, int q_cols, int kv_cols, int Hkv, int D, int page,
                            void* stream) {
  if (gemm_bf16_checks(a, lda, w, ldw, act, accumulate, out_dtype, ldo, M, N, K)) return 1;
  if (kv_cache) {
    DA_REQUIRE(out_dtype == DA_BF16 && !accumulate && q_cols >= 0 && kv_cols == Hkv * D && q_cols + 2 * kv_cols == N &&
               page > 0 && (page & (page - 1)) == 0, "gemm_bf16: the q|k|v columns (%d + 2*%d) must add up to N=%d, the page size a power of two", q_cols, kv_cols, N);
  }
  if (M == 0) return 0;
  const Epilogue ep{bias, bias_dtype, act, accumulate, out, out_dtype, ldo};
  const KvScatter kv{kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page};
  return gemm_bf16_launch(a, lda, w, ldw, ep, kv, M, N, K, stream);
}

// The same for few rows (da_gemm_few_rows) of a q | k | v | rest product whose values have a size of their own and whose
// columns behind v are not kept (see KvScatter).
extern "C" int da_gemm_bf16_kv_split(const void* a, int lda, const void* w, int ldw, const void* bias, int bias_dtype, void* out,
                                     int ldo, int M, int N, int K, void* kv_cache, const int* slot_map, int q_cols, int Hkv, int D,
                                     int Dv, int page, void* stream) {
  if (gemm_bf16_checks(a, lda, w, ldw, DA_ACT_NONE, 0, DA_BF16, ldo, M, N, K)) return 1;
  DA_REQUIRE(da_gemm_few_rows(M, N), "gemm_bf16_kv_split: %d rows of %d columns are more than the kernels for few rows take", M, N);
  DA_REQUIRE(kv_cache && slot_map && q_cols >= 0 && Hkv > 0 && D > 0 && Dv > 0 && page > 0 && q_cols + Hkv * (D + Dv) <= N,
             "gemm_bf16_kv_split: the k and v columns leave the row");
  if (M == 0) return 0;
  const Epilogue ep{bias, bias_dtype, DA_ACT_NONE, 0, out, DA_BF16, ldo};
  const KvScatter kv{kv_cache, slot_map, q_cols, Hkv * D, Hkv, D, page, Dv};
  return gemm_bf16_launch(a, lda, w, ldw, ep, kv, M, N, K, stream);
}

static int gemm_bf16_launch(const void* a, int lda, const void* w, int ldw, const Epilogue& ep, const KvScatter& kv, int M, int N,
                            int K, void* stream) {
  const int act = ep.act, accumulate = ep.accumulate, out_dtype = ep.out_dtype;
  hipStream_t s = (hipStream_t)stream;
  const bf16_t* A = (const bf16_t*)a;
  const bf16_t* W = (const bf16_t*)w;
  if (sk4_takes(M, N, K)) {
    launch_skinny4(s, A, lda, W, ldw, ep, kv, M, N, K);
  } else if (da_gemm_few_rows(M, N)) {
    const int nw = sk_wavefronts(N, K);
    if (nw == 4 ? launch_skinny<4>(s, A, lda, W, ldw, ep, kv, M, N, K)
                : (nw == 8 ? launch_skinny<8>(s, A, lda, W, ldw, ep, kv, M, N, K)
                           : launch_skinny<12>(s, A, lda, W, ldw, ep, kv, M, N, K))) return 1;
  } else {
    // Smaller tiles where larger ones would leave compute units idle (measured on GPT-2's shapes).
    // Every configuration sums a row's products in the same order (64-wide slabs, 16 at a time), so
    // the choice does not change a result; but for the deep tiles, whose wavefronts share k out.
    const bool direct = da_gemm_wide_takes(act, accumulate, out_dtype, K);       // (into the stream: without an activation)
    const int deep = direct && accumulate ? da_gemm_deep_choice(M, N, K) : DA_WIDE_NONE;
    if (deep != DA_WIDE_NONE) {
      da_gemm_wide_launch(s, A, lda, W, ldw, ep, kv, M, N, K, deep);
      DA_CHECK_LAUNCH("gemm_bf16");
      return 0;
    }
    const int wide = direct ? da_gemm_wide_choice(M, N, K) : DA_WIDE_NONE;
    if (wide != DA_WIDE_NONE) {
      // operands straight into LDS where such tiles fill the chip: the same sums in the same order, less LDS traffic
      da_gemm_wide_launch(s, A, lda, W, ldw, ep, kv, M, N, K, wide);
      DA_CHECK_LAUNCH("gemm_bf16");
      return 0;
    }
    const long tiles128 = (long)da_ceil_div(M, 128) * da_ceil_div(N, 128);
    const long tiles12864 = (long)da_ceil_div(M, 128) * da_ceil_div(N, 64);
    // (up to 256 tiles a workgroup has its compute unit to itself: four slabs in flight instead of two, with the
    // registers that a second workgroup would have needed; into the stream, with whole slabs of K, the deep tiles are in front)
    if (tiles128 >= 192 && tiles128 <= 256) launch_tile<128, 128, 4, 2, 4>(s, A, lda, W, ldw, ep, kv, M, N, K);
    else if (tiles128 >= 192) launch_tile<128, 128, 4, 2, 2>(s, A, lda, W, ldw, ep, kv, M, N, K);
    else if (tiles12864 >= 192) launch_tile<128, 64, 4, 2, 4>(s, A, lda, W, ldw, ep, kv, M, N, K);
    else launch_tile<64, 64, 2, 2, 4>(s, A, lda, W, ldw, ep, kv, M, N, K);
  }
  DA_CHECK_LAUNCH("gemm_bf16");
  return 0;
}

// out = a @ w[group of the row].T on the block tiles: rows come in groups of `group_rows` (128 or a multiple), group i
// uses the matrix w + tile_group[i] * group_stride elements ([N, K] each), groups with a negative entry are skipped.
// The same tiles and the same order of sums as da_gemm_bf16's.
extern "C" int da_gemm_bf16_grouped(const void* a, int lda, const void* w, int ldw, long group_stride,
                                    const int* tile_group, int group_rows, void* out, int out_dtype, int ldo, int M,
                                    int N, int K, void* stream, int act) {
  DA_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_bf16_grouped: bad sizes M=%d N=%d K=%d", M, N, K);
  DA_REQUIRE(K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0 && group_stride % 8 == 0,
             "gemm_bf16_grouped: K, lda, ldw and the stride between matrices must be multiples of 8");
  DA_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_bf16_grouped: operands must be 16-byte aligned");
  DA_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm_bf16_grouped: leading sizes too small");
  DA_REQUIRE(tile_group && group_rows > 0 && group_rows % 128 == 0 && M % group_rows == 0,
             "gemm_bf16_grouped: %d rows in groups of %d (a multiple of 128 that divides the rows)", M, group_rows);
  DA_REQUIRE(out_dtype == DA_BF16 || out_dtype == DA_F32, "gemm_bf16_grouped: bad output dtype");
  DA_REQUIRE(act >= DA_ACT_NONE && act <= DA_ACT_LAST, "gemm_bf16_grouped: unknown activation %d", act);
  if (M == 0) return 0;
  Epilogue ep{nullptr, 0, act, 0, out, out_dtype, ldo};
  KvScatter kv{nullptr, nullptr, 0, 0, 0, 0, 0};
  Grouping gr{tile_group, group_stride, group_rows};
  hipStream_t s = (hipStream_t)stream;
  const long tiles128 = (long)da_ceil_div(M, 128) * da_ceil_div(N, 128);
  if (tiles128 >= 192) launch_tile<128, 128, 4, 2, 2>(s, (const bf16_t*)a, lda, (const bf16_t*)w, ldw, ep, kv, M, N, K, gr);
  else launch_tile<128, 64, 4, 2, 4>(s, (const bf16_t*)a, lda, (const bf16_t*)w, ldw, ep, kv, M, N, K, gr);
  DA_CHECK_LAUNCH("gemm_bf16_grouped");
  return 0;
}
