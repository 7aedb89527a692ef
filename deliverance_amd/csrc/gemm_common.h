// Shared by the matrix-core products: fragment types, the epilogue, 16-byte loads.
#pragma once
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

struct Epilogue {
  const void* bias;
  int bias_dtype;
  int act;
  int accumulate;
  void* out;
  int out_dtype;
  int ldo;
};

// The products of few rows take pointers and sizes first, as single arguments: the first 14 words are in registers when a wavefront
// starts (build.py: KERNARG_PRELOAD).  A structure among a kernel's arguments never is, so an Epilogue comes in two parts.
struct EpilogueRest {
  int bias_dtype, act, accumulate, out_dtype;
};
static inline EpilogueRest epilogue_rest(const Epilogue& ep) { return EpilogueRest{ep.bias_dtype, ep.act, ep.accumulate, ep.out_dtype}; }

__device__ __forceinline__ void epilogue_store(const Epilogue& ep, int m, int n, float v, float bias) {
  v = ep.out_dtype == DA_BF16 ? apply_act_bf16(v + bias, ep.act) : apply_act(v + bias, ep.act);
  const size_t o = (size_t)m * ep.ldo + n;
  if (ep.accumulate) ((float*)ep.out)[o] += v;
  else if (ep.out_dtype == DA_BF16) ((bf16_t*)ep.out)[o] = f32_to_bf16(v);
  else ((float*)ep.out)[o] = v;
}

// A product's k shared out over workgroups (blockIdx.y: the share, k_share of K each): share s stores its sums, without bias or
// activation, in rows of their own behind those of share s - 1; whoever reads the rows next adds them up (da_layernorm_join).
__device__ __forceinline__ void gemm_take_share(const bf16_t* __restrict__& a, const bf16_t* __restrict__& w, Epilogue& ep, int M, int& K, int k_share) {
  const int k0 = (int)blockIdx.y * k_share;
  a += k0;
  w += k0;
  ep.out = (float*)ep.out + (size_t)blockIdx.y * M * ep.ldo;
  K = K - k0 < k_share ? K - k0 : k_share;
}

// For a fused q|k|v projection: the k and v columns of a row also go to the row's place in the
// paged cache (keys row-major, values dimension-major; see common.h).
struct KvScatter {
  void* cache;          // null: no scatter
  const int* slot_map;  // per row: page * page_size + row in page, or -1
  int q_cols, kv_cols;  // k occupies columns [q_cols, q_cols + kv_cols), v the next kv_cols
  int Hkv, D, page;
  // The products for few rows also take values of a size of their own (a page then holds Hkv * page * D keys, then Hkv *
  // Dv * page values) and columns behind q | k | v that are not kept; 0: Dv is D, and v is the last of the columns.
  int Dv = 0;
};

// column n (>= q_cols) of a row whose place in the cache is row `row` of page `pg`
__device__ __forceinline__ void kv_scatter_bits(const KvScatter& kv, int pg, int row, int n, bf16_t bits) {
  const int c2 = n - kv.q_cols, is_v = c2 >= kv.kv_cols, cc = is_v ? c2 - kv.kv_cols : c2;
  const int h = cc / kv.D, d = cc % kv.D;
  bf16_t* cache = (bf16_t*)kv.cache;
  if (is_v) cache[cache_v_base(pg, h, kv.Hkv, kv.page, kv.D) + (long long)d * kv.page + row] = bits;
  else cache[cache_k_row(pg, h, row, kv.Hkv, kv.page, kv.D) + d] = bits;
}

// x / d for numbers that are the same for the whole wavefront's divisor (x >= 0): head and page sizes are nearly always powers of two,
// and the general division is some forty instructions of a chain that everything waits for.
__device__ __forceinline__ int div_uniform(int x, int d) { return (d & (d - 1)) == 0 ? x >> (31 - __builtin_clz(d)) : x / d; }

// Where column n of a row goes in its page: entry `at` of the page for the page's first row, `step` entries further for each row
// behind it (0: the column is not kept, `at` is no place).  It needs no row, so kernels work it out while their operands are on the way.
struct KvColumn {
  long long at;
  int step;
};
__device__ __forceinline__ KvColumn kv_column(const KvScatter& kv, int n) {
  const int c = n - kv.q_cols, cv = c - kv.kv_cols, Dv = kv.Dv ? kv.Dv : kv.D;
  if (c < 0) return KvColumn{0, 0};
  if (cv < 0) return KvColumn{c + (long long)div_uniform(c, kv.D) * (kv.page - 1) * kv.D, kv.D};
  return KvColumn{((long long)kv.Hkv * kv.D + cv) * kv.page, cv < kv.Hkv * Dv ? 1 : 0};
}
// (a column that is not kept is left out here, and not by each caller: its `at` may lie behind the page)
template <typename T = bf16_t>
__device__ __forceinline__ void kv_column_store(const KvScatter& kv, const KvColumn& col, int slot, float v) {
  if (col.step == 0 || slot < 0) return;
  const int pg = div_uniform(slot, kv.page), row = slot - pg * kv.page;
  from_f32((T*)kv.cache + (pg * ((long long)kv.Hkv * kv.page * (kv.D + (kv.Dv ? kv.Dv : kv.D))) + col.at + (long long)row * col.step), v);
}

// The values of 32 rows of a product whose k and v columns go to the cache.  Values are dimension-major: 4 rows whose places
// are 4 consecutive ones from a multiple of 4 on are 8 consecutive bytes.  A lane of the accumulators holds the rows 4 i ..
// 4 i + 3 of its column.  `slot` is the place of row `lane % 32` (-1: none); the answers
// are the same for each half of the wavefront.
//  - kv_all_runs: all rows are in such groups and the groups begin with row 0 (what one prompt portion's rows are, asked
//    first): stored from the accumulators, 8 bytes a group.
//  - kv_run_offset: all groups begin with row 1, 2 or 3 (a prompt behind another one of odd length): stored from the parked
//    tile, a column a lane (kv_store_values32).
//  - else (rows of several sequences, places in any order, rows without a place): from the accumulators again, group by
//    group, entry by entry where a group is no run (kv_store_run).
// The first way has code of its own, without a look at each group: inside a step, where another kernel's code has taken the
// instruction cache, a q|k|v product of 2,048 rows, N = 4,800, K = 1,600 takes 46.7 us with it and 48.7 where the first and
// the last share theirs.
// Up to 512 rows the second way is not taken: fewer tiles than compute units store their values entry by entry in less time
// than the chain through LDS takes (prompts of odd lengths, K = 768, N = 2,304: 552 rows 12.2 us against 11.7, 300 rows
// with one group a turn 8.9 against 10.3; K = 1,600, N = 4,800: 23.0 against 18.6, 17.0 against 16.7).
#define KV_WALK_MIN_ROWS 513
#define KV_WAY_RUNS 4
__device__ __forceinline__ bool kv_all_runs(int slot, int lane) {
  const int first = dpp_move_i<0x00, 0xF>(slot, slot);      // quad_perm [0, 0, 0, 0]
  const uint64_t off = __builtin_amdgcn_ballot_w64(first < 0 || (first & 3) != 0 || slot != first + (lane & 3));
  return (uint32_t)(off >> (lane & 32)) == 0;
}
// 4 consecutive rows' values of one column (in w): su holds the rows' places
__device__ __forceinline__ void kv_store_run(bf16_t* col, const uint4& su, uint2 w, bool vwide, long long page_stride, int lgp, int pmask) {
  const struct { int x, y, z, w; } sl = {(int)su.x, (int)su.y, (int)su.z, (int)su.w};
  if (vwide && sl.x >= 0 && (sl.x & 3) == 0 && sl.y == sl.x + 1 && sl.z == sl.x + 2 && sl.w == sl.x + 3) {
    *(uint2*)(col + (long long)(sl.x >> lgp) * page_stride + (sl.x & pmask)) = w;
    return;
  }
  const int s4[4] = {sl.x, sl.y, sl.z, sl.w};
  const uint32_t w2[2] = {w.x, w.y};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (s4[e] >= 0) col[(long long)(s4[e] >> lgp) * page_stride + (s4[e] & pmask)] = (bf16_t)(w2[e / 2] >> (16 * (e % 2)));
}
// Which row the groups begin with: 1 .. 3, or 0 where they do not; the two halves of the wavefront may hold two pieces.
__device__ __forceinline__ int kv_run_offset(int slot, int lane) {
  const int half = lane & 32, r = lane & 31;
  const int s0 = half ? __builtin_amdgcn_readlane(slot, 32) : __builtin_amdgcn_readlane(slot, 0), o = (4 - (s0 & 3)) & 3;
  const int base = o + ((r - o) & ~3);                  // (arithmetic: rows before the first group have a base below 0)
  const bool whole = base >= 0 && base + 3 < 32;
  const int first = __shfl(slot, half + (whole ? base : r), DA_WAVE);
  const uint64_t off = __builtin_amdgcn_ballot_w64(whole && (slot < 0 || (first & 3) != 0 || slot != first + (r - base)));
  return (uint32_t)(off >> half) ? 0 : o;
}

// A column a lane: `park` is the lane's entry of the first row in LDS (rows LDT entries apart), `dst` the lane's column's
// run in page 0 (null: not a value column).  Seven groups from row `offset` (1 .. 3) on, two a turn, 8 bytes each; the 4 rows
// outside of them are stored one by one.  (A prompt behind another one of odd length begins
// anywhere in a tile: stored entry by entry from the accumulators its values took half as long as the product, 1,624 rows,
// N = 3,072, K = 1,024 32.0 us against 23.8; the same rows in whole groups of 4 21.9.  Rows without such groups are no
// faster from here: 552 rows of prompts of 21 tokens, N = 3,072, K = 1,024 15.2 us against 13.6.  The loop stays a loop: with
// every offset written out the code is so long that also prompts that never run it wait, 2,048 rows, N = 4,800, K = 1,600
// between a step's other kernels 48.9 -> 52.0.)
template <int LDT>
__device__ __forceinline__ void kv_store_values32(const bf16_t* park, int slot, int offset, bf16_t* dst, long long page_stride, int lgp, int pmask) {
#pragma unroll 1
  for (int g = 0; g < 7; g += 2) {                      // (the last one is stored twice)
    const int r0 = offset + 4 * g, r1 = offset + 4 * min(g + 1, 6);
    const bf16_t *const p = park + r0 * LDT, *const q = park + r1 * LDT;
    const uint32_t p0 = p[0], p1 = p[LDT], p2 = p[2 * LDT], p3 = p[3 * LDT], q0 = q[0], q1 = q[LDT], q2 = q[2 * LDT], q3 = q[3 * LDT];
    const int s0 = __builtin_amdgcn_readlane(slot, r0), s1 = __builtin_amdgcn_readlane(slot, r1);
    if (dst) {
      *(uint2*)(dst + (long long)(s0 >> lgp) * page_stride + (s0 & pmask)) = make_uint2(p0 | (p1 << 16), p2 | (p3 << 16));
      *(uint2*)(dst + (long long)(s1 >> lgp) * page_stride + (s1 & pmask)) = make_uint2(q0 | (q1 << 16), q2 | (q3 << 16));
    }
  }
  int sl[4];
  bf16_t v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = e < offset ? e : 28 + e;
    sl[e] = __builtin_amdgcn_readlane(slot, r);
    v[e] = park[r * LDT];
  }
  if (dst)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (sl[e] >= 0) dst[(long long)(sl[e] >> lgp) * page_stride + (sl[e] & pmask)] = v[e];
}

__device__ __forceinline__ uint4 load16(const bf16_t* p) { return *(const uint4*)p; }


// The tiles whose operands go from memory straight into LDS (gemm_wide.hip): what they take, which of their
// shapes pays for a product's sizes (DA_WIDE_NONE: none), and their launch.
enum { DA_WIDE_NONE = -1, DA_WIDE_256x256 = 0, DA_WIDE_256x128 = 1, DA_WIDE_128x128 = 2, DA_DEEP_128x128 = 3, DA_DEEP_128x64 = 4 };
#define DA_DEEP_MIN_K 1024
bool da_gemm_wide_takes(int act, int accumulate, int out_dtype, int K);
extern "C" int da_gemm_wide_choice(int M, int N, int K);
extern "C" int da_gemm_deep_choice(int M, int N, int K);
void da_gemm_wide_launch(hipStream_t s, const bf16_t* A, int lda, const bf16_t* W, int ldw, const Epilogue& ep,
                         const KvScatter& kv, int M, int N, int K, int shape, int k_share = 0);
