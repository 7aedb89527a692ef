// The block-tile product for large steps: operands from memory straight into LDS.
//
//   out[m, n] (+)= act( sum_k a[m, k] * w[n, k] + bias[n] )        (a [M, K], w [N, K], bfloat16, K contiguous)
//
// The first shape: tiles of 256 x 256, eight wavefronts, two a SIMD, each with 128 x 64 of the tile (4 x 2
// products of 32 x 32 x 16, 128 accumulation registers): a k-step of 16 takes 6 fragment reads for 8 matrix
// instructions, half the LDS traffic a flop of the 128 x 128 tile kernel (gemm_mfma.hip), whose matrix cores
// wait for LDS most of the time.  Two smaller shapes for products whose 256 x 256 tiles would leave compute
// units idle, both with eight wavefronts: 256 x 128 (64 x 64 a wavefront: 4 reads for 4 matrix instructions),
// and 128 x 128 (32 x 64 a wavefront), of which two workgroups share a compute unit (da_gemm_wide_choice).
// A slab of 64 elements of k is 128 bytes a row, one cache line: it goes from memory into LDS
// without passing registers (da_lds_dma.h), into one of two stages for a (one slab ahead of the
// products) and one of three for w (two slabs ahead: weights come from memory, not from a cache); one
// barrier a slab.  Rows lie unpadded in LDS (a copy writes 1,024 consecutive bytes: 8 rows); the
// 16-byte pieces of row r are stored at position piece ^ (r / 2 % 8), which the copy does by choosing what
// each lane fetches, so that the fragment reads of 16 consecutive rows spread over all banks.
// Fragments are read one k-step ahead of the products that use them.
//
// An output element of gemm_wide_kernel sums over k in ascending steps of 16 like the forms of gemm_mfma.hip's
// tiles: the result has the same bits.  (gemm_deep_kernel, further down, shares k out inside a workgroup: two or
// four such sums, added.)  K must be a multiple of 64 (other sizes go to gemm_mfma.hip's kernels).
//
// The epilogue is per wavefront: 32 rows x 64 columns at a time are parked in the wavefront's own piece
// of LDS (bias and activation applied, rounded to the output's type), and leave in 16-byte pieces, whole
// rows side by side; += adds to 16-byte pieces read the same way; a fused q|k|v projection also writes
// its k and v columns to the rows' places in the paged cache (keys in 16-byte pieces of their rows,
// values in 8-byte runs where 4 rows' places are consecutive: kv_all_runs).
#include "gemm_common.h"
#include <da_lds_dma.h>
#include <da_read_arg.h>
#include <type_traits>

#define WD_BK 64
#define WD_ROW_BYTES (WD_BK * 2)
#define WD_REGION_BYTES 8960          // a wavefront's piece of LDS in the epilogue: 32 x 68 floats, then 32 places

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// OUTMODE: 0 bf16 store, 1 f32 store, 2 f32 +=
template <int TM, int TN, int ACT, int OUTMODE>
__device__ __forceinline__ void
wide_epilogue(floatx16 (&acc)[TM][TN], const float (&bias)[TN], char* region, const void* safe, const Epilogue& ep,
              const KvScatter& kv, int M, int N, int mw, int nw, int lane) {
  constexpr int WC = 32 * TN;                                   // the wavefront's columns
  constexpr int ES = OUTMODE == 0 ? 2 : 4, CH = 16 / ES;       // bytes an element; elements a 16-byte piece
  constexpr int LDT = WC + CH;                                  // a parked row, padded by one piece
  constexpr int CPR = WC / CH, NCHK = 32 * CPR / 64;            // pieces a row; pieces a lane and pass
  static_assert(32 * LDT * ES + 32 * 4 <= WD_REGION_BYTES, "a wavefront's epilogue region");
  const int fr = lane % 32;
  int* slots = (int*)(region + 32 * LDT * ES);
  const bool wide = (uintptr_t)ep.out % 16 == 0 && ep.ldo % CH == 0;
  // A q|k|v product's cache write: what does not change from pass to pass.  The page size is a power of two
  // (checked on the host): places split into page and row by shift and mask.
  const int lgp = kv.cache ? 31 - __builtin_clz(kv.page) : 0, pmask = kv.page - 1;
  const int v0 = kv.q_cols + kv.kv_cols;                        // the first value column
  const bool kwide = kv.cache && (uintptr_t)kv.cache % 16 == 0 && kv.D % 8 == 0 && kv.q_cols % 8 == 0;
  const bool vwide = kv.cache && (uintptr_t)kv.cache % 8 == 0 && kv.page % 4 == 0;
  const long long page_stride = 2LL * kv.Hkv * kv.page * kv.D;
  int kh[NCHK], kd[NCHK];                                       // head and dimension of a key piece's first column
  int vcol[TN];                                                 // a value column's place in a page: its head's values, its dimension's run
  if (OUTMODE == 0 && kv.cache) {
#pragma unroll
    for (int k = 0; k < NCHK; ++k) {
      const int c2 = nw + ((lane + 64 * k) % CPR) * CH - kv.q_cols, cs = c2 > 0 ? c2 : 0;
      kh[k] = cs / kv.D;
      kd[k] = cs % kv.D;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int cc = nw + j * 32 + fr - v0, cs = cc > 0 ? cc : 0;
      vcol[j] = (kv.Hkv + cs / kv.D) * kv.page * kv.D + (cs % kv.D) * kv.page;
    }
  }
  // the places of every pass's rows (row `lane % 32` of each) are asked for here: a load inside a pass would wait for the
  // stores of the pass before it
  int sl[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = mw + i * 32 + fr;
    sl[i] = OUTMODE == 0 && kv.cache ? *(m < M ? kv.slot_map + m : (const int*)safe) : -1;
    sl[i] = m < M ? sl[i] : -1;
  }
  // (a pass per constant i: an index that is not a constant would put the accumulators into memory)
  auto pass = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const int mp = mw + i * 32;                                 // the pass's first row
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int ml = 8 * (r / 4) + 4 * (lane / 32) + (r % 4), nl = j * 32 + fr;
        if (OUTMODE == 0) ((bf16_t*)region)[ml * LDT + nl] = f32_to_bf16(apply_act_bf16(acc[i][j][r] + bias[j], ACT));
        else ((float*)region)[ml * LDT + nl] = apply_act(acc[i][j][r] + bias[j], ACT);
      }
    if (OUTMODE == 0 && kv.cache && lane < 32) slots[lane] = sl[i];
    wave_lds_sync();

    uint4 val[NCHK];
    int mm[NCHK], nn[NCHK];
#pragma unroll
    for (int k = 0; k < NCHK; ++k) {
      const int q = lane + 64 * k, row = q / CPR, c = q % CPR;
      mm[k] = mp + row;
      nn[k] = nw + c * CH;
      val[k] = *(const uint4*)(region + (size_t)(row * LDT + c * CH) * ES);
    }
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
    // (for +=, such a piece still holds the bare products here: only whole pieces were added to above)
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

    if (OUTMODE == 0 && kv.cache) {
      // keys: eight dimensions of one key are one piece of its cache row (head and dimension of a piece's
      // columns were worked out before the passes)
#pragma unroll
      for (int k = 0; k < NCHK; ++k) {
        const int slot = slots[mm[k] - mp];
        if (slot < 0 || nn[k] >= N || nn[k] + 8 <= kv.q_cols || nn[k] >= v0) continue;
        const int pg = slot >> lgp, prow = slot & pmask;
        if (kwide) {
          *(uint4*)((bf16_t*)kv.cache + cache_k_row(pg, kh[k], prow, kv.Hkv, kv.page, kv.D) + kd[k]) = val[k];
          continue;
        }
        const uint32_t words[4] = {val[k].x, val[k].y, val[k].z, val[k].w};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (nn[k] + e >= kv.q_cols && nn[k] + e < v0)
            kv_scatter_bits(kv, pg, prow, nn[k] + e, (bf16_t)(words[e / 2] >> (16 * (e % 2))));
      }
      // values: straight from the accumulators (a lane holds 4 consecutive rows of its column, r % 4; the lane of the
      // other half holds the 4 rows beside them), or from LDS, a column a lane; see kv_all_runs
      if (nw + WC > v0) {
        bf16_t* vb = (bf16_t*)kv.cache;
        int offset = 0;
        const bool runs = vwide && __builtin_amdgcn_readfirstlane(kv_all_runs(sl[i], lane));
        if (__builtin_expect(runs, 1)) {
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const int n = nw + j * 32 + fr;
            if (n < v0 || n >= N) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              uint32_t w2[2];
#pragma unroll
              for (int e = 0; e < 2; ++e)
                w2[e] = pack2_bf16(apply_act_bf16(acc[i][j][4 * q + 2 * e] + bias[j], ACT),
                                   apply_act_bf16(acc[i][j][4 * q + 2 * e + 1] + bias[j], ACT));
              const int s0 = slots[8 * q + 4 * (lane / 32)];
              *(uint2*)(vb + vcol[j] + (long long)(s0 >> lgp) * page_stride + (s0 & pmask)) = make_uint2(w2[0], w2[1]);
            }
          }
        } else if (!(vwide && M >= KV_WALK_MIN_ROWS && (offset = __builtin_amdgcn_readfirstlane(kv_run_offset(sl[i], lane))) != 0)) {
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const int n = nw + j * 32 + fr;
            if (n < v0 || n >= N) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              uint32_t w2[2];
#pragma unroll
              for (int e = 0; e < 2; ++e)
                w2[e] = pack2_bf16(apply_act_bf16(acc[i][j][4 * q + 2 * e] + bias[j], ACT),
                                   apply_act_bf16(acc[i][j][4 * q + 2 * e + 1] + bias[j], ACT));
              kv_store_run(vb + vcol[j], *(const uint4*)&slots[8 * q + 4 * (lane / 32)], make_uint2(w2[0], w2[1]), vwide, page_stride, lgp, pmask);
            }
          }
        } else {
          static_assert(WC == 64, "a column a lane");
          const int n = nw + lane, cc = n - v0;
          bf16_t* const dst = cc >= 0 && n < N ? vb + (long long)(kv.Hkv + cc / kv.D) * kv.page * kv.D + (cc % kv.D) * kv.page : nullptr;
          kv_store_values32<LDT>((const bf16_t*)region + lane, sl[i], offset, dst, page_stride, lgp, pmask);
        }
      }
    }
    wave_lds_sync();       // the next pass parks over what this one read
  };
  pass(std::integral_constant<int, 0>{});
  if (TM > 1) pass(std::integral_constant<int, (TM > 1 ? 1 : 0)>{});
  if (TM > 2) pass(std::integral_constant<int, (TM > 2 ? 2 : 0)>{});
  if (TM > 3) pass(std::integral_constant<int, (TM > 3 ? 3 : 0)>{});
}

// BM x BN: the tile; WM x WN wavefronts of (BM / WM) x (BN / WN) each.  In use: 256 x 256 with 2 x 4
// wavefronts of 128 x 64, one workgroup a compute unit (160 KB of LDS); 256 x 128 with 4 x 2 of 64 x 64
// (112 KB); 128 x 128 with 4 x 2 of 32 x 64, two workgroups a compute unit (80 KB each); which of them
// for which sizes: da_gemm_wide_choice.  Measured beside them: 256 x 256 with four wavefronts of 128 x 128
// (a third less LDS traffic; 15 to 25 % slower: one wavefront a SIMD has nobody to fill its waits);
// 128 x 128 with 2 x 2 wavefronts of 64 x 64 (7 to 10 % behind the eight wavefronts at a short K).
template <int BM, int BN, int WM, int WN, int ACT, int OUTMODE>
__global__ void __launch_bounds__(WM * WN * 64)
gemm_wide_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const void* bias_p, int lda, int ldw, int M, int N, int K,
                 int tiles_m, int tiles_n, int k_share, int bias_dtype, void* out, int ldo, KvScatter kv) {
  // (the first 14 words are in registers when the wavefront starts)
  Epilogue ep{bias_p, bias_dtype, ACT, OUTMODE == 2, out, OUTMODE == 0 ? DA_BF16 : DA_F32, ldo};
  gemm_take_share(a, w, ep, M, K, k_share);
  // Two stages of a slab of a, three of a slab of w.  The rows of a were written by the kernel before and
  // come from a cache; w comes from memory for the first time and needs the longer way ahead.
  constexpr int A_BYTES = BM * WD_ROW_BYTES, W_BYTES = BN * WD_ROW_BYTES;      // a slab of a, of w, in LDS
  constexpr int NW = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int CA = BM / 8 / NW, CW = BN / 8 / NW;                             // copies a wavefront and slab
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && BM % (32 * WM) == 0 && BN % (32 * WN) == 0 && NW % 2 == 0,
                "the tile does not split over the wavefronts");
  static_assert(BN / WN == 64, "the epilogue parks 64 columns a wavefront");
  __shared__ __attribute__((aligned(1024))) char smem[2 * A_BYTES + 3 * W_BYTES];
  static_assert(NW * WD_REGION_BYTES <= 2 * A_BYTES + 3 * W_BYTES, "the epilogue regions fit the stages");
  char* const smem_a = smem;
  char* const smem_w = smem + 2 * A_BYTES;

  // Each XCD (workgroups that follow each other in launch order land on different ones) takes a
  // contiguous run of tiles, m fastest, so that its workgroups share slabs of w in its L2.
  const int nblocks = tiles_m * tiles_n;
  int pid = blockIdx.x;
  {
    const int per = nblocks / 8, rem = nblocks % 8;
    const int xcd = pid % 8, local = pid / 8;
    pid = xcd * per + (xcd < rem ? xcd : rem) + local;
  }
  const int m0 = (pid % tiles_m) * BM, n0 = (pid / tiles_m) * BN;

  const int t = threadIdx.x, lane = t % 64;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
  const int fr = lane % 32, fk = lane / 32;

  // Copies: a stage of a (of w) is BM / 8 (BN / 8) blocks of 8 rows; wavefront v takes blocks v, v + NW, ...
  // Lane l of a copy stands for row l / 8 of the block and position l % 8 of that row, which holds the
  // row's piece (l % 8) ^ (r / 2 % 8), r the row's number in the stage.  Rows past the edge of a or w read
  // the last row: what they give is never stored.
  const bf16_t* src_a[CA];
  const bf16_t* src_w[CW];
  int blk[CA > CW ? CA : CW];                        // byte offset of the wavefront's blocks in a stage
  {
    // (row r of a stage is row l / 8 of block v + NW i, NW even: r / 2 % 8 = (4 (v % 2) + l / 16) % 8)
    const int rl = lane / 8, piece = (lane % 8) ^ ((4 * (wave & 1) + (rl >> 1)) & 7);
#pragma unroll
    for (int i = 0; i < (CA > CW ? CA : CW); ++i) {
      const int b = i * NW + wave;
      const int ra = m0 + b * 8 + rl, rw = n0 + b * 8 + rl;
      if (i < CA) src_a[i] = a + (size_t)(ra < M ? ra : M - 1) * lda + piece * 8;
      if (i < CW) src_w[i] = w + (size_t)(rw < N ? rw : N - 1) * ldw + piece * 8;
      blk[i] = b * 1024;
    }
  }
#define WD_COPY_A(i, stage) { lds_dma16(src_a[i], smem_a + (stage) * A_BYTES + blk[i]); src_a[i] += WD_BK; }
#define WD_COPY_W(i, stage) { lds_dma16(src_w[i], smem_w + (stage) * W_BYTES + blk[i]); src_w[i] += WD_BK; }

  // Fragments: lane l gives row l % 32 of a 32-row piece and the 8 k from 8 * (l / 32) of a k-step:
  // piece 2 * step + l / 32 of its row, stored at that number ^ (row / 2 % 8).
  int a_off[TM], w_off[TN], k_off[4];
#pragma unroll
  for (int i = 0; i < TM; ++i) a_off[i] = (wm + i * 32 + fr) * WD_ROW_BYTES;
#pragma unroll
  for (int j = 0; j < TN; ++j) w_off[j] = (wn + j * 32 + fr) * WD_ROW_BYTES;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) k_off[ks] = ((2 * ks + fk) ^ ((fr >> 1) & 7)) * 16;
#define WD_READ(FA, FB, sa, sw, ks)                                                                                  \
  {                                                                                                                  \
    const char* pa = smem_a + (sa) * A_BYTES + k_off[ks];                                                            \
    const char* pw = smem_w + (sw) * W_BYTES + k_off[ks];                                                            \
    _Pragma("unroll") for (int i = 0; i < TM; ++i) FA[i] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(pa + a_off[i])); \
    _Pragma("unroll") for (int j = 0; j < TN; ++j) FB[j] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(pw + w_off[j])); \
  }
#define WD_MFMA1(FA, FB, q) \
  acc[(q) / TN][(q) % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(FA[(q) / TN], FB[(q) % TN], acc[(q) / TN][(q) % TN], 0, 0, 0)
#define WD_MFMA(FA, FB) { _Pragma("unroll") for (int q = 0; q < TM * TN; ++q) WD_MFMA1(FA, FB, q); }
#define WD_FENCE() __builtin_amdgcn_sched_barrier(0)

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // Order of the copies: a(0) w(0) | a(1) w(1) | w(2) | then, after the barrier that ends slab s, a(s + 2)
  // and w(s + 3) into the stages that slab s left.  Copies land in the order they were asked for, so
  // "slab s + 1 is there" is "at most the four youngest copies, w(s + 2), are still under way".
  const int nslab = K / WD_BK;
  bf16x8_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];
#pragma unroll
  for (int i = 0; i < CA; ++i) WD_COPY_A(i, 0);
#pragma unroll
  for (int i = 0; i < CW; ++i) WD_COPY_W(i, 0);
  if (nslab > 1) {
#pragma unroll
    for (int i = 0; i < CA; ++i) WD_COPY_A(i, 1);
#pragma unroll
    for (int i = 0; i < CW; ++i) WD_COPY_W(i, 1);
  }
  if (nslab > 2) {
#pragma unroll
    for (int i = 0; i < CW; ++i) WD_COPY_W(i, 2);
  }
  // The bias is asked for behind the first slabs, as raw bits from a place that always exists (the waits below count copies: with the
  // bias's loads among the youngest they wait for a copy or two more than they need, once), with the arguments that only the epilogue
  // uses.  No other ordinary load stands between here and the end of the slabs.
  const bool bias_bf16 = ep.bias_dtype == DA_BF16;
  uint32_t braw[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 32 + fr;
    const bool has = ep.bias && n < N;
    const void* bsrc = has ? ep.bias : (const void*)w;
    const int idx = has ? n : 0;
    braw[j] = bias_bf16 ? (uint32_t)((const bf16_t*)bsrc)[idx] : ((const uint32_t*)bsrc)[idx];
  }
  da_read_arg(ep.out);
  da_read_arg(ep.ldo);
  if (OUTMODE == 0) {
    da_read_arg(kv.cache);
    da_read_arg(kv.q_cols);
    da_read_arg(kv.Hkv);
    da_read_arg(kv.page);
  }
  static_assert(CA + 2 * CW <= 15, "the count of copies under way fits its field");
  if (nslab > 2) DA_WAIT_VMCNT(CA + 2 * CW); else if (nslab > 1) DA_WAIT_VMCNT(CA + CW); else DA_WAIT_VMCNT(0);
  __builtin_amdgcn_s_barrier();
  WD_READ(fa0, fb0, 0, 0, 0);
  int sw = 0;                                          // the stage of w that holds slab s
  // One slab.  COPY_A: slab s + 2 exists; COPY_W: slab s + 3 exists; NEXT: slab s + 1 exists.
  auto slab = [&](int s, auto copy_a_c, auto copy_w_c, auto next_c) {
    constexpr bool COPY_A = decltype(copy_a_c)::value, COPY_W = decltype(copy_w_c)::value, NEXT = decltype(next_c)::value;
    const int sa = s & 1, sw1 = sw == 2 ? 0 : sw + 1;
    WD_FENCE();
    // (the first product stands in front of the reads: the wait that the compiler puts before it then
    // covers the fragments it needs and nothing that was only just asked for)
    WD_MFMA1(fa0, fb0, 0);
    WD_FENCE();
    WD_READ(fa1, fb1, sa, sw, 1);
    WD_FENCE();
#pragma unroll
    for (int q = 1; q < TM * TN; ++q) WD_MFMA1(fa0, fb0, q);
    WD_FENCE();
    WD_READ(fa0, fb0, sa, sw, 2);
    WD_FENCE();
    WD_MFMA(fa1, fb1);
    WD_FENCE();
    WD_READ(fa1, fb1, sa, sw, 3);
    WD_FENCE();
    WD_MFMA(fa0, fb0);
    WD_FENCE();
    // Slab s + 1 must have landed, and every wavefront must be done reading slab s, before a(s + 2) and
    // w(s + 3) take its place: one barrier for both.
    if (COPY_A) DA_WAIT_VMCNT(CW); else DA_WAIT_VMCNT(0);     // (COPY_A: the tail before this one asked for w(s + 2) last)
    __builtin_amdgcn_s_waitcnt(0xC07F);                        // lgkmcnt(0): this wavefront's reads of slab s are complete
    __builtin_amdgcn_s_barrier();
    // The slab's last k-step, its products one by one, and between them the copies and the reads of slab
    // s + 1's first fragments: the matrix cores have work while the wavefront issues the rest.
    constexpr int CPQ = (CA + CW + TM * TN - 1) / (TM * TN);      // copies after each product
    constexpr int RPQ = (TM + TN + TM * TN - 1) / (TM * TN);      // reads after each product
#pragma unroll
    for (int q = 0; q < TM * TN; ++q) {
      WD_MFMA1(fa1, fb1, q);
#pragma unroll
      for (int c = q * CPQ; c < (q + 1) * CPQ; ++c) {             // (all of a's before all of w's)
        if (COPY_A && c < CA) WD_COPY_A(c, sa);
        if (COPY_W && c >= CA && c < CA + CW) WD_COPY_W(c - CA, sw);
      }
#pragma unroll
      for (int r = q * RPQ; r < (q + 1) * RPQ; ++r) {             // (a's fragments, then w's)
        constexpr int LAST_A = TM - 1, LAST_W = TN - 1;
        const int ia = r < TM ? r : LAST_A, iw = (r >= TM && r < TM + TN) ? r - TM : LAST_W;    // (indices that exist, whatever r)
        if (NEXT && r < TM) fa0[ia] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(smem_a + (sa ^ 1) * A_BYTES + k_off[0] + a_off[ia]));
        if (NEXT && r >= TM && r < TM + TN) fb0[iw] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(smem_w + sw1 * W_BYTES + k_off[0] + w_off[iw]));
      }
      WD_FENCE();
    }
    sw = sw1;
  };
  {
    const std::true_type yes{};
    const std::false_type no{};
    int s = 0;
    for (; s + 3 < nslab; ++s) slab(s, yes, yes, yes);
    if (s + 2 < nslab) slab(s++, yes, no, yes);
    if (s + 1 < nslab) slab(s++, no, no, yes);
    slab(s, no, no, no);
  }
#undef WD_COPY_A
#undef WD_COPY_W
#undef WD_READ
#undef WD_MFMA
#undef WD_MFMA1
#undef WD_FENCE
  float bias[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) bias[j] = !ep.bias ? 0.f : (bias_bf16 ? __uint_as_float(braw[j] << 16) : __uint_as_float(braw[j]));
  // (the last barrier of the loop: nobody reads the stages any more)
  wide_epilogue<TM, TN, ACT, OUTMODE>(acc, bias, smem + wave * WD_REGION_BYTES, (const void*)w, ep, kv, M, N, m0 + wm, n0 + wn, lane);
}

// Which tile a workgroup takes.  Workgroups that follow each other in launch order land on different dies (8, each with an L2 of its
// own), and what a die reads of a and w it reads from behind its L2 once: with 2^lg_m blocks of tiles by rows and 8 / 2^lg_m by
// columns, a die a block, as few rows and columns as the shape allows.  Where the blocks' sizes differ so much that a die would have a
// round of tiles more (DIE_RUNS), runs of tiles, rows first, as gemm_wide_kernel has them.  False: no tile for this workgroup.
// (1,624 rows, N = 1,024, K = 4,096 and 1,024 in a step, the mean of the two in a profiled run: runs 20.7 us, blocks 20.1.)
#define DIE_RUNS 4
__device__ __forceinline__ bool die_tile(int id, int tiles_m, int tiles_n, int lg_m, int& tile_m, int& tile_n) {
  const int die = id % 8, local = id / 8;
  if (lg_m == DIE_RUNS) {
    const int n = tiles_m * tiles_n, per = n / 8, rem = n % 8, pid = die * per + (die < rem ? die : rem) + local;
    tile_n = pid / tiles_m;
    tile_m = pid - tile_n * tiles_m;
    return local < per + (die < rem ? 1 : 0);
  }
  const int xm = die & ((1 << lg_m) - 1), xn = die >> lg_m, lg_n = 3 - lg_m;
  const int m_lo = (xm * tiles_m) >> lg_m, m_n = (((xm + 1) * tiles_m) >> lg_m) - m_lo;
  const int n_lo = (xn * tiles_n) >> lg_n, n_n = (((xn + 1) * tiles_n) >> lg_n) - n_lo;
  if (local >= m_n * n_n) return false;
  const int q = local / m_n;
  tile_m = m_lo + local - q * m_n;
  tile_n = n_lo + q;
  return true;
}
struct DieCut { int lg_m, workgroups; };
static DieCut die_cut(int tiles_m, int tiles_n, int bm, int bn) {
  const long tiles = (long)tiles_m * tiles_n;
  const int rounds = da_ceil_div(da_ceil_div(tiles, 8), 32);          // of 32 compute units a die
  DieCut best{DIE_RUNS, (int)tiles};
  long least = 0;
  for (int lg = 0; lg <= 3; ++lg) {
    const int m = da_ceil_div(tiles_m, 1 << lg), n = da_ceil_div(tiles_n, 8 >> lg);
    if (da_ceil_div((long)m * n, 32) > rounds) continue;
    const long rows = (long)m * bm + (long)n * bn;
    if (best.lg_m == DIE_RUNS || rows < least) { best = DieCut{lg, 8 * m * n}; least = rows; }
  }
  return best;
}

// ---------------------------------------------------------------------------------------------
// Products into the residual stream that leave a tile or less to a compute unit: k shared out inside the workgroup.
//
// A compute unit pulls 62 to 68 GB/s out of L2 whatever is in flight (tiles of 128 x 128 and 128 x 64, one a compute unit, one to five
// slabs ahead, copies alone: 2,048 rows, N = 1,600, K = 6,400 52 us; 1,624 rows, N = 1,024, K = 4,096 24 us), so the tile is given and
// what is left is to keep that stream going.  The tiles of gemm_mfma.hip at these sizes wait for LDS instead: their wavefronts of 32 x 64
// (32 x 32) read 96 KB (64) of fragments for a slab of 32 (24) KB.  Here a wavefront has 64 x 64 of the tile and KG wavefronts share a
// position, each with every KG-th k-step: 64 KB (32) a slab, and eight wavefronts to hide each other's waits all the same.  Operands go
// straight into LDS, S slabs ahead (all of LDS: a workgroup a compute unit); a wavefront's fragments of the next slab are read between
// this slab's products; one barrier a slab, after which the stage it stands for is free.  The wavefronts of a position leave their sums
// in LDS, and the first of them add them up in order of k-steps, 32 rows each: an element is KG sums, each in ascending k, added one to the other.
// us, recorded one behind the other, cold weights, gemm_mfma.hip's tiles -> this: 2,048 rows, N = 1,600, K = 6,400 63.6 -> 60.7 (691 TFLOP/s), 1,624 rows,
// N = 1,024, K = 4,096 27.0 -> 22.5 (605); error against 64 bits 4.9e-7 -> 3.4e-7 and 3.8e-7 -> 1.8e-7.
// ---------------------------------------------------------------------------------------------
template <int BM, int BN, int KG, int S>
__global__ void __launch_bounds__(512)
gemm_deep_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const void* bias_p, int lda, int ldw, int M, int N, int K,
                 int tiles, int lg_m, int ldo, int bias_dtype, float* out) {
  constexpr int NW = 8, WM = BM / 64, WN = BN / 64, TM = 2, TN = 2, KS = 4 / KG;      // k-steps of a slab a wavefront
  static_assert(WM * WN * KG == NW && KS >= 1 && KG >= 2, "eight wavefronts");
  constexpr int A_BYTES = BM * WD_ROW_BYTES, STAGE = A_BYTES + BN * WD_ROW_BYTES;
  constexpr int CA = BM / 8 / NW, CW = BN / 8 / NW, C = CA + CW;                      // copies a wavefront and slab
  static_assert(C * (S - 1) <= 63, "the count of copies under way fits its field");
  constexpr int SUM_BYTES = WM * WN * TM * TN * (KG - 1) * 4096;
  static_assert(SUM_BYTES + TM * WM * WN * WD_REGION_BYTES <= S * STAGE, "the wavefronts' sums and the epilogue's regions fit the stages");
  __shared__ __attribute__((aligned(1024))) char smem[S * STAGE];

  int tile_m, tile_n;
  if (!die_tile(blockIdx.x, tiles & 0xffff, tiles >> 16, lg_m, tile_m, tile_n)) return;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int t = threadIdx.x, lane = t % 64, wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int kg = wave / (WM * WN), pos = wave % (WM * WN), wm = (pos % WM) * 64, wn = (pos / WM) * 64;
  const int fr = lane % 32, fk = lane / 32;

  const bf16_t* src[C];
  int dst[C];
  {
    const int rl = lane / 8, piece = (lane % 8) ^ ((4 * (wave & 1) + (rl >> 1)) & 7);   // (rows lie in LDS as in gemm_wide_kernel)
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int b = (i < CA ? i : i - CA) * NW + wave, r = (i < CA ? m0 : n0) + b * 8 + rl;
      src[i] = (i < CA ? a + (size_t)(r < M ? r : M - 1) * lda : w + (size_t)(r < N ? r : N - 1) * ldw) + piece * 8;
      dst[i] = (i < CA ? 0 : A_BYTES) + b * 1024;
    }
  }
  int a_off[TM], w_off[TN], k_off[KS];
#pragma unroll
  for (int i = 0; i < TM; ++i) a_off[i] = (wm + i * 32 + fr) * WD_ROW_BYTES;
#pragma unroll
  for (int j = 0; j < TN; ++j) w_off[j] = A_BYTES + (wn + j * 32 + fr) * WD_ROW_BYTES;
#pragma unroll
  for (int i = 0; i < KS; ++i) k_off[i] = ((2 * (kg + i * KG) + fk) ^ ((fr >> 1) & 7)) * 16;

  auto copy = [&](int stage) {
#pragma unroll
    for (int i = 0; i < C; ++i) {
      lds_dma16(src[i], smem + stage * STAGE + dst[i]);
      src[i] += WD_BK;
    }
  };
  struct Frags { bf16x8_t a[KS][TM], w[KS][TN]; };
  auto read1 = [&](Frags& f, int stage, int q) {                     // fragment q of a slab's KS (TM + TN)
    const char* const p = smem + stage * STAGE;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
#pragma unroll
      for (int x = 0; x < TM; ++x)
        if (q == i * (TM + TN) + x) f.a[i][x] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(p + k_off[i] + a_off[x]));
#pragma unroll
      for (int x = 0; x < TN; ++x)
        if (q == i * (TM + TN) + TM + x) f.w[i][x] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(p + k_off[i] + w_off[x]));
    }
  };
  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nslab = K / WD_BK;                                        // S at least (checked on the host)
#pragma unroll
  for (int i = 0; i < S; ++i) copy(i);
  const bool bias_bf16 = bias_dtype == DA_BF16;
  uint32_t braw[TN];                                                  // (behind the first copies: as in gemm_wide_kernel)
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 32 + fr;
    const bool has = bias_p && n < N;
    const void* bsrc = has ? bias_p : (const void*)w;
    braw[j] = bias_bf16 ? (uint32_t)((const bf16_t*)bsrc)[has ? n : 0] : ((const uint32_t*)bsrc)[has ? n : 0];
  }
  da_read_arg(out);
  DA_WAIT_VMCNT6(C * (S - 1));
  __builtin_amdgcn_s_barrier();
  Frags f0, f1;
#pragma unroll
  for (int q = 0; q < KS * (TM + TN); ++q) read1(f0, 0, q);
  int stage = 0;                                                      // slab s's
  // Slab s: its fragments are in `now` when the barrier is passed, slab s + 1 is in LDS, and stage s % S is free.  LEFT: slabs behind s + 1
  // that may still be under way; COPY: slab s + S exists; NEXT: slab s + 1 does.
  auto slab = [&](Frags& now, Frags& next, auto left_c, auto copy_c, auto next_c) {
    constexpr int LEFT = decltype(left_c)::value;
    constexpr bool COPY = decltype(copy_c)::value, NEXT = decltype(next_c)::value;
    const int after = stage + 1 == S ? 0 : stage + 1;
    if (NEXT) {
      DA_WAIT_VMCNT6(C * LEFT);
      __builtin_amdgcn_s_waitcnt(0xC07F);                            // lgkmcnt(0): slab s's fragments have arrived
      __builtin_amdgcn_s_barrier();
      if (COPY) copy(stage);
    }
    __builtin_amdgcn_sched_barrier(0);
    constexpr int NQ = KS * TM * TN;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      constexpr int TT = TM * TN;
      const int i = q / TT, x = q % TT / TN, y = q % TN;
      acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(now.a[i][x], now.w[i][y], acc[x][y], 0, 0, 0);
      if (NEXT && q < KS * (TM + TN)) read1(next, after, q);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(NQ >= KS * (TM + TN), "a read behind each product");
    stage = after;
  };
  {
    const std::true_type yes{};
    const std::false_type no{};
    const std::integral_constant<int, S - 2> steady{};
    int s = 0;
    for (; s + 1 < nslab - S; s += 2) {
      slab(f0, f1, steady, yes, yes);
      slab(f1, f0, steady, yes, yes);
    }
    // the last S slabs, whose copies are all asked for
    auto tail = [&](Frags& x, Frags& y) {
      slab(x, y, std::integral_constant<int, S - 2>{}, no, yes);
      if constexpr (S >= 3) slab(y, x, std::integral_constant<int, S - 3>{}, no, yes);
      if constexpr (S >= 4) slab(x, y, std::integral_constant<int, S >= 4 ? S - 4 : 0>{}, no, yes);
      if constexpr (S >= 5) slab(y, x, std::integral_constant<int, S >= 5 ? S - 5 : 0>{}, no, yes);
      if constexpr (S >= 6) slab(x, y, std::integral_constant<int, S >= 6 ? S - 6 : 0>{}, no, yes);
      static_assert(S >= 5 && S <= 6, "the tail is written out for five and six stages");
      if constexpr (S == 5) slab(x, y, std::integral_constant<int, 0>{}, no, no);
      else slab(y, x, std::integral_constant<int, 0>{}, no, no);
    };
    if (s < nslab - S) {
      slab(f0, f1, steady, yes, yes);
      tail(f1, f0);
    } else tail(f0, f1);
  }
  float bias[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) bias[j] = !bias_p ? 0.f : (bias_bf16 ? __uint_as_float(braw[j] << 16) : __uint_as_float(braw[j]));
  // the sums of a position's wavefronts meet: wavefront kg < TM owns the rows 32 kg .. of it; a wavefront leaves in LDS what it does not own
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();                                       // (nobody reads the stages any more)
  float* const sums = (float*)smem;
  auto place = [&](int x, int g, int y) { return sums + ((((x * (KG - 1) + (g > x ? g - 1 : g)) * WM * WN + pos) * TN + y) * 16) * 64 + lane; };
#pragma unroll
  for (int x = 0; x < TM; ++x)
    if (kg != x) {
#pragma unroll
      for (int y = 0; y < TN; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r) place(x, kg, y)[r * 64] = acc[x][y][r];
    }
  lds_barrier();
  if (kg >= TM) return;
  floatx16 sum[1][TN];
  auto add = [&](auto xc) {
    constexpr int x = decltype(xc)::value;
#pragma unroll
    for (int y = 0; y < TN; ++y)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = x == 0 ? acc[x][y][r] : place(x, 0, y)[r * 64];
#pragma unroll
        for (int g = 1; g < KG; ++g) v += g == x ? acc[x][y][r] : place(x, g, y)[r * 64];
        sum[0][y][r] = v;
      }
  };
  if (kg == 0) add(std::integral_constant<int, 0>{});
  else add(std::integral_constant<int, 1>{});
  const Epilogue ep{bias_p, bias_dtype, DA_ACT_NONE, 1, out, DA_F32, ldo};
  const KvScatter kv{nullptr, nullptr, 0, 0, 0, 0, 0};
  wide_epilogue<1, TN, DA_ACT_NONE, 2>(sum, bias, smem + SUM_BYTES + wave * WD_REGION_BYTES, (const void*)w, ep, kv, M, N, m0 + wm + 32 * kg, n0 + wn, lane);
}

template <int BM, int BN, int KG, int S>
static void launch_deep(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep, int M, int N, int K) {
  const int tiles_m = da_ceil_div(M, BM), tiles_n = da_ceil_div(N, BN);
  const DieCut cut = die_cut(tiles_m, tiles_n, BM, BN);
  hipLaunchKernelGGL((gemm_deep_kernel<BM, BN, KG, S>), dim3(cut.workgroups), dim3(512), 0, s, A, W, ep.bias, lda, ldw, M, N, K,
                     tiles_m | tiles_n << 16, cut.lg_m, ep.ldo, ep.bias_dtype, (float*)ep.out);
}

template <int BM, int BN, int WM, int WN, int ACT>
static void launch_wide_act(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep,
                            const KvScatter& kv, int M, int N, int K, int k_share) {
  const int tiles_m = da_ceil_div(M, BM), tiles_n = da_ceil_div(N, BN);
  const dim3 grid(tiles_m * tiles_n, da_ceil_div(K, k_share)), block(WM * WN * 64);
  if (ep.accumulate)
    hipLaunchKernelGGL((gemm_wide_kernel<BM, BN, WM, WN, DA_ACT_NONE, 2>), grid, block, 0, s, A, W, ep.bias, lda, ldw, M, N, K, tiles_m, tiles_n, k_share, ep.bias_dtype, ep.out, ep.ldo, kv);
  else if (ep.out_dtype == DA_F32)
    hipLaunchKernelGGL((gemm_wide_kernel<BM, BN, WM, WN, DA_ACT_NONE, 1>), grid, block, 0, s, A, W, ep.bias, lda, ldw, M, N, K, tiles_m, tiles_n, k_share, ep.bias_dtype, ep.out, ep.ldo, kv);
  else
    hipLaunchKernelGGL((gemm_wide_kernel<BM, BN, WM, WN, ACT, 0>), grid, block, 0, s, A, W, ep.bias, lda, ldw, M, N, K, tiles_m, tiles_n, k_share, ep.bias_dtype, ep.out, ep.ldo, kv);
}

template <int BM, int BN, int WM, int WN>
static void launch_wide(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep,
                        const KvScatter& kv, int M, int N, int K, int k_share) {
  switch (ep.act) {
    case DA_ACT_GELU_TANH: launch_wide_act<BM, BN, WM, WN, DA_ACT_GELU_TANH>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share); break;
    case DA_ACT_GELU_ERF: launch_wide_act<BM, BN, WM, WN, DA_ACT_GELU_ERF>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share); break;
    case DA_ACT_RELU: launch_wide_act<BM, BN, WM, WN, DA_ACT_RELU>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share); break;
    case DA_ACT_SILU: launch_wide_act<BM, BN, WM, WN, DA_ACT_SILU>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share); break;
    case DA_ACT_RELU2: launch_wide_act<BM, BN, WM, WN, DA_ACT_RELU2>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share); break;
    default: launch_wide_act<BM, BN, WM, WN, DA_ACT_NONE>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share); break;
  }
}

// What these tiles take: K in whole slabs, and an activation only with a bfloat16 result (the forms
// that a model's layers use; everything else stays with gemm_mfma.hip's tiles).
bool da_gemm_wide_takes(int act, int accumulate, int out_dtype, int K) {
  return K % WD_BK == 0 && K >= WD_BK && (act == DA_ACT_NONE || (!accumulate && out_dtype == DA_BF16));
}

// Which shape of tile pays, if any (DA_WIDE_NONE: gemm_mfma.hip's tiles).  A tile is a compute unit's
// work for the whole product, so the tiles must fill most of the last round of 256 compute units.
// Measured on MI355X with 512 to 8,192 rows, N from 768 to 6,400, K from 768 to 6,400, stores and +=:
//  - 256 x 256 where its tiles fill 55 % of their last round: ahead of the 128 x 128 tiles from 152 tiles on
//    (2,048 rows, N = 4,800: 39 against 47 us; N = 6,400, 200 tiles: 42 against 62 us), behind at 128 tiles
//    and fewer (N = 4,096: 30 against 27 us);
//  - else, where 128 x 128 tiles would be 257 to 512, so that some compute units had two of gemm_mfma.hip's
//    and others one: up to a K of 2,048 tiles of 256 x 128, one a compute unit (2,048 rows: N = 2,304,
//    K = 768 16.2 against 18.9 us; N = 3,072, K = 1,024 20.3 against 23.3; 1,536 rows, N = 4,800, K = 1,600
//    28.8 against 35.3); beyond, 128 x 128, two a compute unit (4,096 rows, N = 1,600, K = 6,400, += 113
//    against 130 us; 8,192 rows, N = 768, K = 3,072 58 against 69);
//  - where they would be 140 to 256, one a compute unit: 128 x 128 up to a K of 4,096 (1,024 rows, N = 2,304
//    10.6 against 13.5 us; 512 rows, N = 4,800 16.7 against 22.3; 2,048 rows, N = K = 1,600, += 21.1 against
//    23.3; 4,096 rows, N = 1,024, K = 4,096 48.6 against 56.4); beyond, the four slabs in flight of
//    gemm_mfma.hip's tiles win (2,048 rows, N = 1,600, K = 6,400: 65 against 79 us).
// Into the stream the deep tiles are asked first (da_gemm_deep_choice): of what adds, the third line decides for K below 3,072
// and between 3,072 and 4,096 for stores alone.
int da_gemm_wide_choice(int M, int N, int K) {
  const long tiles = (long)da_ceil_div(M, 256) * da_ceil_div(N, 256);
  const long rounds = (tiles + 255) / 256;
  if (tiles * 100 >= rounds * 256 * 55) return DA_WIDE_256x256;
  const long tiles128 = (long)da_ceil_div(M, 128) * da_ceil_div(N, 128);
  if (tiles128 > 256 && tiles128 <= 512) return K <= 2048 ? DA_WIDE_256x128 : DA_WIDE_128x128;
  if (tiles128 >= 140 && tiles128 <= 256 && K <= 4096) return DA_WIDE_128x128;
  return DA_WIDE_NONE;
}

// Which of the deep tiles a product into the stream takes, if any: those that are one a compute unit at most, where the tiles that the
// other forms have are more than that, or wait for LDS.  Measured on MI355X with cold weights, recorded side by side, about 320 sizes with N from 512 to 8,192 and
// K from 1,024 to 8,192, us, other forms / deep:
//  - 128 x 64 where there are up to 256 of them and tiles of 64 x 64 would be more: 1,624 rows, N = 1,024, K = 4,096 27.0 / 22.5, K = 1,024
//    10.9 / 10.4; 1,300 rows, K = 4,096 29.2 / 21.7; 900 rows, N = K = 2,048 16.9 / 16.0; 2,048 rows, N = 768, K = 3,072 22.1 / 18.9.  Where tiles of
//    64 x 64 are one a compute unit themselves they stay (1,024 rows, N = 1,024, K = 4,096, 256 of them: 20.2 / 22.0).  So do the other forms in two places
//    where they are level: K = 1,024 with 192 tiles and more of 2,048 columns and more (700 rows, N = 2,048 9.9 / 10.0, 715 rows, N = 2,560 10.7 / 10.9, 354 rows,
//    N = 5,120 11.0 / 10.9; with 1,535 rows, N = 1,216 11.4 / 11.0, with K = 1,152, 593 rows, N = 2,560 11.3 / 10.3), and more than 16 tiles by rows whose
//    blocks do not fit the dies (a die then reads nearly all rows: die_tile; 2,600 rows, N = 768, K = 1,024 12.2 / 12.6, K = 3,072 25.0 / 25.0, 2,107 rows, N = 896, K = 1,088
//    12.4 / 12.2, 3,442 rows, N = 576, K = 1,024 13.7 / 14.5; with 13 tiles by rows, 1,549 rows, N = 1,152, K = 2,048 17.0 / 15.7);
//  - 128 x 128 where there are up to 256 of them and of 128 x 64 more, K from 3,072: 2,048 rows, N = 1,600, K = 6,400 63.6 / 60.7, 1,624 rows
//    74.4 / 56.2; 4,096 rows, N = 1,024, K = 4,096 47.4 / 41.0 (gemm_wide_kernel's 128 x 128); 2,048 rows, N = 1,536, K = 3,072 33.3 / 32.8; 1,300 rows, N = 2,048, K = 8,192
//    91.8 / 60.4.  (K = 2,048: 4,096 rows, N = 1,024 26.1 / 27.1; two rounds of them: 4,096 rows, N = 2,048, K = 4,096 84.6 / 102.5.)
extern "C" int da_gemm_deep_choice(int M, int N, int K) {
  if (K % WD_BK || K < DA_DEEP_MIN_K) return DA_WIDE_NONE;
  const int rows128 = da_ceil_div(M, 128), cols64 = da_ceil_div(N, 64);
  const long t64 = (long)da_ceil_div(M, 64) * cols64, t12864 = (long)rows128 * cols64;
  if (t12864 > 256) return K >= 3072 && (long)rows128 * da_ceil_div(N, 128) <= 256 ? DA_DEEP_128x128 : DA_WIDE_NONE;
  if (t64 <= 256 || (K <= 1024 && t12864 >= 192 && N >= 2048)) return DA_WIDE_NONE;
  return rows128 > 16 && die_cut(rows128, cols64, 128, 64).lg_m == DIE_RUNS ? DA_WIDE_NONE : DA_DEEP_128x64;
}

void da_gemm_wide_launch(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep,
                         const KvScatter& kv, int M, int N, int K, int shape, int k_share) {
  if (k_share <= 0) k_share = K;
  if (shape == DA_DEEP_128x128 || shape == DA_DEEP_128x64) {          // (up to 32,767 tiles each way: checked where a shape is asked for)
    if (shape == DA_DEEP_128x128) launch_deep<128, 128, 2, 5>(s, A, lda, W, ldw, ep, M, N, K);
    else launch_deep<128, 64, 4, 6>(s, A, lda, W, ldw, ep, M, N, K);
    return;
  }
  if (shape == DA_WIDE_128x128) launch_wide<128, 128, 4, 2>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share);
  else if (shape == DA_WIDE_256x128) launch_wide<256, 128, 4, 2>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share);
  else launch_wide<256, 256, 2, 4>(s, A, lda, W, ldw, ep, kv, M, N, K, k_share);
}

// These tiles alone, of the shape asked for (DA_WIDE_256x256, DA_WIDE_256x128, DA_WIDE_128x128), whatever the
// product's sizes (tests and timing call it; da_gemm_bf16 chooses by them).
extern "C" int da_gemm_bf16_wide(const void* a, int lda, const void* w, int ldw, const void* bias, int bias_dtype,
                                 int act, int accumulate, void* out, int out_dtype, int ldo, int M, int N, int K,
                                 void* kv_cache, const int* slot_map, int q_cols, int kv_cols, int Hkv, int D, int page,
                                 int shape, void* stream) {
  DA_REQUIRE(shape >= DA_WIDE_256x256 && shape <= DA_DEEP_128x64, "gemm_bf16_wide: unknown tile shape %d", shape);
  DA_REQUIRE(shape <= DA_WIDE_128x128 || (accumulate && !kv_cache && K >= DA_DEEP_MIN_K), "gemm_bf16_wide: this shape adds into the stream, K from %d on", DA_DEEP_MIN_K);
  DA_REQUIRE(shape <= DA_WIDE_128x128 || (da_ceil_div(M, 128) < 32768 && da_ceil_div(N, 64) < 32768), "gemm_bf16_wide: too many tiles for this shape");
  DA_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_bf16_wide: bad sizes M=%d N=%d K=%d", M, N, K);
  DA_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K && ldo >= N, "gemm_bf16_wide: leading sizes (lda=%d ldw=%d ldo=%d)", lda, ldw, ldo);
  DA_REQUIRE(((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0), "gemm_bf16_wide: operands must be 16-byte aligned");
  DA_REQUIRE(!accumulate || out_dtype == DA_F32, "gemm_bf16_wide: accumulation needs a 32-bit output");
  DA_REQUIRE(act >= DA_ACT_NONE && act <= DA_ACT_LAST, "gemm_bf16_wide: unknown activation %d", act);
  DA_REQUIRE(da_gemm_wide_takes(act, accumulate, out_dtype, K),
             "gemm_bf16_wide: K=%d must be a multiple of %d, and an activation goes with a bfloat16 result", K, WD_BK);
  if (kv_cache) {
    DA_REQUIRE(out_dtype == DA_BF16 && !accumulate && q_cols >= 0 && kv_cols == Hkv * D && q_cols + 2 * kv_cols == N &&
               page > 0 && (page & (page - 1)) == 0, "gemm_bf16_wide: the q|k|v columns (%d + 2*%d) must add up to N=%d, the page size a power of two", q_cols, kv_cols, N);
  }
  Epilogue ep{bias, bias_dtype, act, accumulate, out, out_dtype, ldo};
  KvScatter kv{kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page};
  da_gemm_wide_launch((hipStream_t)stream, (const bf16_t*)a, lda, (const bf16_t*)w, ldw, ep, kv, M, N, K, shape);
  DA_CHECK_LAUNCH("gemm_bf16_wide");
  return 0;
}
