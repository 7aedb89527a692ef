// Paged attention for prompt portions in bfloat16 on the matrix cores (flash-style: scores never
// leave the chip).  A portion's rows sit at positions past .. past+T-1 of their sequence; row i
// sees the keys lo_i .. past+i of the cache (earlier steps' keys and the portion's own, which were
// written just before).
//
// One workgroup per (portion, query head, 32 * W query rows); W wavefronts of 32 rows each.  Keys
// come in aligned tiles of 64 through two LDS buffers, two tiles ahead in registers: the key rows as they lie in the pages, the values as
// they lie in the pages too (dimension-major: a row of the LDS tile is one dimension, 64 keys).
// Per tile and wavefront, with MFMA 32x32x16:
//   S^T[key, row] = K . Q^T          keys are the MFMA's rows, so one lane holds ONE query row's
//                                     scores for 16 keys: row maximum and sum need one exchange
//                                     (lane ^ 32) instead of a reduction over the wavefront;
//   online softmax in 32-bit (maximum, exp, sum, rescale: the recurrence of
//   native/src/main/resources/decode_paged_attention_f32.wgsl:31-65);
//   O^T[dim, row] += V^T . P^T       P^T is already in registers in the layout of the B operand
//                                     (the matching, permuted order of keys is used for V^T).
// Formulas: core/src/main/java/io/teknek/deliverance/generator/CausalSelfAttention.java:458-502.
// A row's sums run over key tiles in ascending order starting at the aligned tile of its lo: the
// order depends on the row's position (and window) only.
//
// Few workgroups (a prompt of a thousand tokens and a dozen heads gives fewer than the chip has
// compute units, and the one with the last rows walks all keys alone): the wavefronts of a
// workgroup then also share out the keys.  RB row blocks of 32 x KP key phases: a round parks KP
// consecutive tiles in KP LDS buffers, wavefront (row block, phase k) multiplies tile k of the round,
// and at the end the phases' partial results (maximum, sum of weights, weighted sum) are merged in
// LDS in the order of the phases.  A tile's phase is (first key / 64) mod KP, whatever the workgroup:
// a row's sums still depend on its position, the window and KP only; RB x KP is chosen from the
// step's shape on the host.  Smaller row blocks are for short portions only: every row block of 32
// reads its keys anew, and on long prompts that traffic, not the longest workgroup, binds.
//
// Compiled a second time with PF_REL (attn_prefill_rel.hip) the kernel also takes what some designs put on the
// scores: a bias by the distance between query and key (a table [Hq][n_dist], 32-bit, the last entry for every
// larger distance; the head's row sits in LDS, times log2 e) and a query temperature
// 1 + t_coef * ln(floor((p + 1) / t_every) + 1) that multiplies the row's scale (a lane owns one query row).
// A tile whose keys all lie n_dist - 1 or more behind the wavefront's first row adds one constant.  The plain
// build has none of that code.
#include "common.h"
#include <da_lane_swap.h>
#include <da_read_arg.h>
#include <type_traits>

#ifdef PF_REL
#define PF_KERNEL attn_prefill_rel_kernel
#define PF_REL_MAX_DIST 1024       // entries of the bias row that the workgroup keeps in LDS
#define PF_REL_PAD 96              // a tile's keys reach at most 59 + 35 distances past either end of the row
#define PF_REL_PARAMS , const float* __restrict__ rel_bias, int n_dist, float t_coef, int t_every
#define PF_REL_ARGS , rel_bias, n_dist, t_coef, t_every
#else
#define PF_KERNEL attn_prefill_kernel
#define PF_REL_PARAMS
#define PF_REL_ARGS
#endif

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

#define PF_BK 64           // keys per tile
#define PF_VLD (PF_BK + 8) // padded length of a value row in LDS
#define PF_BT_MAX 2048      // block-table entries a workgroup keeps in LDS (more are read from memory)
#define PF_BT_MAX_PHASED 512   // ... where key phases need the LDS for their tiles
#define PF_PHASED_MAX_WORKGROUPS 256   // 128-row workgroups up to which eight wavefronts (4 x 2) are ahead of four: one a compute unit

// head size / 16; wavefronts (32 query rows each) per workgroup; whether the block table's entries
// for the workgroup's keys fit its LDS copy (a table entry read from memory in front of a tile's loads
// makes them wait for it, and for every load still in flight)
// Included by attn_both.hip (DA_ATTN_BODIES) the kernel is a function that is told which workgroup it is.
// Q_LATE: the rows of q are asked for behind the first tile's keys and values (pf_q_late below says where)
template <int D16, int RB, int KP, bool BT_LDS, bool Q_LATE>
#ifdef DA_ATTN_BODIES
#define PF_SEQ pf_seq
#define PF_BLOCK pf_block
#define PF_BLOCKS pf_blocks
__device__ __forceinline__ void
attn_prefill_body(int pf_seq, int h, int pf_block, int pf_blocks,
#else
#define PF_SEQ (int)blockIdx.y
#define PF_BLOCK (int)blockIdx.z
#define PF_BLOCKS (int)gridDim.z
// (head sizes up to 64 with four wavefronts: registers held to 256, so that two workgroups share a compute unit)
__global__ void __launch_bounds__(RB * KP * DA_WAVE, (RB * KP == 4 && D16 <= 4) ? 2 : 1)
PF_KERNEL(
#endif
          const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, const int* __restrict__ block_table,
          const int* __restrict__ q_start, const int* __restrict__ seq_lens, int q_ld, int max_blocks, int Hq, int Hkv, int seq0,
          int page, float scale, int window, bf16_t* __restrict__ out, int out_ld PF_REL_PARAMS) {
#ifndef DA_ATTN_BODIES
  const int h = blockIdx.x;
#endif
  constexpr int D = D16 * 16;
  constexpr int DT = (D + 31) / 32;       // 32-dimension tiles of the output
  constexpr int KLD = D + 8;              // padded length of a key row in LDS
  constexpr int PF_WAVES = RB * KP;
  constexpr int PF_BQ = RB * 32;          // query rows per workgroup
  constexpr int THREADS = PF_WAVES * DA_WAVE;
  // one phase: two buffers, a tile is multiplied out of one while the next is parked in the other;
  // KP phases: the KP tiles of a round
  constexpr int NB = KP == 1 ? 2 : KP;
  constexpr int RT = KP == 1 ? 1 : KP;    // tiles that one fetch asks for
  constexpr int K_PIECES = RT * PF_BK * (D / 8), V_PIECES = RT * DT * 32 * (PF_BK / 8);   // 16-byte pieces of a fetch
  constexpr int NK = (K_PIECES + THREADS - 1) / THREADS, NV = (V_PIECES + THREADS - 1) / THREADS;  // per thread
  constexpr int K_TILE = PF_BK * KLD, V_TILE = DT * 32 * PF_VLD;              // elements of a parked tile
  constexpr int MERGE_FLOATS = (KP - 1) * RB * (DT * 16 + 2) * DA_WAVE;       // the phases' partial results
  constexpr int TILE_BYTES = NB * (K_TILE + V_TILE) * 2;
  __shared__ __attribute__((aligned(16))) char smem[TILE_BYTES > MERGE_FLOATS * 4 ? TILE_BYTES : MERGE_FLOATS * 4];
  bf16_t (*Ks2)[K_TILE] = (bf16_t (*)[K_TILE])smem;
  bf16_t (*Vs2)[V_TILE] = (bf16_t (*)[V_TILE])(smem + NB * K_TILE * 2);
  __shared__ long long bts[KP == 1 ? PF_BT_MAX : PF_BT_MAX_PHASED];   // a page's place in the cache, in bytes
#ifdef PF_REL
  // The head's bias by distance, times log2 e (zeros without a table), in descending order of the distance and
  // with PF_REL_PAD entries beyond both ends (the first and the last value again): a lane's 32 keys of a tile
  // are then 32 fixed places behind one address, and nothing is clamped per key.
  __shared__ float brel[PF_REL_MAX_DIST + 2 * PF_REL_PAD];
#endif

  // The workgroups with the most keys (the last rows) are launched first, those of every (sequence, head) pair
  // before anybody's second-longest: the head and the sequence are the sizes that the dispatcher counts up first.  (Counted the
  // other way round, the long workgroups of the later pairs start when the chip is already full of short ones, and
  // the step ends with a few compute units walking their keys alone: at 2 x 4,096 rows and 12 heads the wavefronts
  // resident over the kernel's time averaged 0.9 a SIMD of 2.)
  const int s = seq0 + PF_SEQ;
  const int row0 = q_start[s], row1 = q_start[s + 1], len = seq_lens[s];
  da_read_arg(scale);
  da_read_arg(out);
  da_read_arg(out_ld);
  const int T = row1 - row0;
  const int i0 = (PF_BLOCKS - 1 - PF_BLOCK) * PF_BQ;
  if (i0 >= T) return;
  const int past = len - T;
  const int hk = Hq == Hkv ? h : h / (Hq / Hkv);
  const int* bt = block_table + (size_t)s * max_blocks;
  const int t = threadIdx.x, lane = t % DA_WAVE, wave = t / DA_WAVE;
  const int col = lane % 32, hf = lane / 32;
  const int rbi = wave % RB, kp = wave / RB;       // the wavefront's row block and key phase
  const int wrow = rbi * 32;

  // this lane's query row (as a column of Q^T) and its position
  const int qi = i0 + wrow + col;
  const bool q_ok = qi < T;
  const int pq = past + qi;
  const int q_lo = (window > 0 && pq - window + 1 > 0) ? pq - window + 1 : 0;
  static_assert(KP == 1 || !Q_LATE, "the forms with phases ask for q at once");
  bf16x8_t qf[D16];
  if (!Q_LATE) {
#pragma unroll
    for (int kd = 0; kd < D16; ++kd) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (q_ok) v = *(const uint4*)(q + (size_t)(row0 + qi) * q_ld + h * D + kd * 16 + hf * 8);
      qf[kd] = __builtin_bit_cast(bf16x8_t, v);
    }
  }
  auto load_q = [&]() {                         // (a column past the portion holds the last row's query; its results are never stored)
    const bf16_t* qr = q + (size_t)(row0 + (q_ok ? qi : T - 1)) * q_ld + h * D + hf * 8;
#pragma unroll
    for (int kd = 0; kd < D16; ++kd) qf[kd] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(qr + kd * 16));
  };
  // the wavefront's rows span positions w_first .. w_last
  const int w_first = past + i0 + wrow;
  const int w_last_row = (i0 + wrow + 31 < T - 1) ? i0 + wrow + 31 : T - 1;
  const bool wave_on = i0 + wrow < T;
  const int w_last = past + w_last_row;
  const int w_lo = (window > 0 && w_first - window + 1 > 0) ? w_first - window + 1 : 0;
  // the workgroup's keys
  const int b_last = past + ((i0 + PF_BQ - 1 < T - 1) ? i0 + PF_BQ - 1 : T - 1);
  const int b_lo = (window > 0 && past + i0 - window + 1 > 0) ? past + i0 - window + 1 : 0;

  floatx16 acc_o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_o[i][r] = 0.f;
  float m = -INFINITY, l = 0.f;                 // running maximum (base-2 domain); sum of the weights of this lane half's keys
#ifdef PF_REL
  // this lane's row has a scale of its own; the bias row is parked before the first barrier below
  const float scale2 = scale * 1.4426950408889634f *
                       (t_every > 0 ? 1.0f + t_coef * logf((float)(((q_ok ? pq : 0) + 1) / t_every + 1)) : 1.0f);
  const int n_rel = rel_bias ? n_dist : 1;
  const int rel_len = n_rel + 2 * PF_REL_PAD;
  for (int i = t; i < rel_len; i += THREADS) {       // place i holds the distance rel_len - 1 - PF_REL_PAD - i
    const int dist = rel_len - 1 - PF_REL_PAD - i, dc = dist < 0 ? 0 : (dist < n_rel ? dist : n_rel - 1);
    brel[i] = rel_bias ? rel_bias[(size_t)h * n_dist + dc] * 1.4426950408889634f : 0.f;
  }
#else
  const float scale2 = scale * 1.4426950408889634f;
#endif

  // The next tile's keys and values are asked for (into registers) before the current tile is
  // multiplied, so their latency hides behind the arithmetic.  Loads are unconditional (a conditional
  // load becomes a branch that serialises them): a key outside b_lo .. b_last reads a key that
  // exists and is replaced by zero.
  // The block table's entries for this workgroup's keys are copied to LDS once: a table entry read
  // from memory in front of every tile would make the tile's loads wait for it, and that wait also
  // drains the loads still in flight for the tiles before.
  const int pg_lo = b_lo >> (31 - __builtin_clz(page)), pg_hi = b_last >> (31 - __builtin_clz(page));
  const long long page_elems = 2LL * Hkv * page * D;
  if (BT_LDS)
    for (int i = t; i <= pg_hi - pg_lo; i += THREADS) bts[i] = bt[pg_lo + i] * page_elems * 2;
  __syncthreads();
  // where a page's keys and values start, in elements from the cache's start
  auto page_at = [&](int key_page) -> long long { return BT_LDS ? bts[key_page - pg_lo] / 2 : bt[key_page] * page_elems; };
  // Two register sets: while a tile is multiplied, the loads of the next two are in flight.
  uint4 rk0[NK], rv0[NV], rk1[NK], rv1[NV];
  const int lg = 31 - __builtin_clz(page);              // page is a power of two (checked on the host)
  const bf16_t* kbase = cache + (long long)hk * page * D;
  const bf16_t* vbase = cache + (long long)(Hkv + hk) * page * D;
  // a tile whose 64 keys all lie in b_lo .. b_last: nothing to clamp, nothing to replace
  // (a fetch covers RT consecutive tiles: key rows kt .. kt + 64 RT - 1; a value piece is 8 keys of
  // one dimension of one tile)
  constexpr int VG = PF_BK / 8, VPT = DT * 32 * VG;       // key groups a tile; value pieces a tile
  // A tile starts at a multiple of 64 keys, a page holds 16, 32 or 64: which page of the tile's pages a thread's
  // piece lies in, and where in that page, never changes.  Both are worked out once; a piece's address is then the
  // page's place (one read of the table in LDS) plus a constant.
  const char* kconst[NK];
  const char* vconst[NV];
  int kpage[NK], vpage[NV];
#pragma unroll
  for (int i = 0; i < NK; ++i) {
    const int c0 = t + i * THREADS, c = c0 < K_PIECES ? c0 : 0;
    const int kr = c / (D / 8), pc = c % (D / 8);
    kpage[i] = kr >> lg;
    kconst[i] = (const char*)(kbase + (kr & (page - 1)) * D + pc * 8);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c0 = t + i * THREADS, c = c0 < V_PIECES ? c0 : 0;
    const int tl = c / VPT, d = (c % VPT) / VG, g = c % VG, k0 = tl * PF_BK + g * 8;
    const int ds = d < D ? d : 0;                        // rows of a padded 32-dimension tile repeat dimension 0
    vpage[i] = k0 >> lg;
    vconst[i] = (const char*)(vbase + ds * page + (k0 & (page - 1)));
  }
  auto page_bytes = [&](int key_page) -> long long { return BT_LDS ? bts[key_page - pg_lo] : bt[key_page] * page_elems * 2; };
  auto fetch_k_fast = [&](uint4* rk, int kt) {
    const int p0 = kt >> lg;
#pragma unroll
    for (int i = 0; i < NK; ++i) rk[i] = *(const uint4*)(kconst[i] + page_bytes(p0 + kpage[i]));
  };
  auto fetch_v_fast = [&](uint4* rv, int kt) {
    const int p0 = kt >> lg;
#pragma unroll
    for (int i = 0; i < NV; ++i) rv[i] = *(const uint4*)(vconst[i] + page_bytes(p0 + vpage[i]));
  };
  auto fetch_fast = [&](uint4* rk, uint4* rv, int kt) {
    fetch_k_fast(rk, kt);
    fetch_v_fast(rv, kt);
  };
  auto fetch_k = [&](uint4* rk, int kt) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int c0 = t + i * THREADS, c = c0 < K_PIECES ? c0 : 0;
      const int kr = c / (D / 8), pc = c % (D / 8), key = kt + kr;
      const bool ok = key >= b_lo && key <= b_last;
      const int ks = ok ? key : b_last;
      rk[i] = *(const uint4*)(kbase + page_at(ks >> lg) + (ks & (page - 1)) * D + pc * 8);
      if (!ok) rk[i] = make_uint4(0, 0, 0, 0);
    }
  };
  auto fetch_v = [&](uint4* rv, int kt) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c0 = t + i * THREADS, c = c0 < V_PIECES ? c0 : 0;
      const int tl = c / VPT, d = (c % VPT) / VG, g = c % VG, key0 = kt + tl * PF_BK + g * 8;   // 8 keys of one dimension
      const bool ok = d < D && key0 + 7 >= b_lo && key0 <= b_last;
      const int ks = ok ? key0 : (b_last / 8) * 8;
      const int ds = d < D ? d : 0;
      uint4 v = *(const uint4*)(vbase + page_at(ks >> lg) + ds * page + (ks & (page - 1)));
      if (!ok) v = make_uint4(0, 0, 0, 0);
      if (key0 < b_lo || key0 + 7 > b_last) {          // rows outside were never written for us
        uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (key0 + e < b_lo || key0 + e > b_last) u[e / 2] &= (e % 2) ? 0x0000ffffu : 0xffff0000u;
        v = make_uint4(u[0], u[1], u[2], u[3]);
      }
      rv[i] = v;
    }
  };
  auto fetch = [&](uint4* rk, uint4* rv, int kt) {
    fetch_k(rk, kt);
    fetch_v(rv, kt);
  };
  // (one phase: the tile goes to buffer `buf`; KP phases: tile k of the fetch goes to buffer k)
  auto stash_k = [&](const uint4* rk, int buf) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int c = t + i * THREADS, kr = c / (D / 8), pc = c % (D / 8);
      if (K_PIECES % THREADS == 0 || c < K_PIECES) *(uint4*)&Ks2[buf + kr / PF_BK][(kr % PF_BK) * KLD + pc * 8] = rk[i];
    }
  };
  auto stash_v = [&](const uint4* rv, int buf) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = t + i * THREADS, tl = c / VPT, d = (c % VPT) / VG, g = c % VG;
      // Within a block of 16 keys a row keeps them in the order 0-3, 8-11, 4-7, 12-15: the 8 keys a lane
      // multiplies at once (4hf.., 8+4hf.., as the scores' registers hold them) are then 16 consecutive
      // bytes, read in one piece and without bank conflicts.
      if (V_PIECES % THREADS == 0 || c < V_PIECES) {
        bf16_t* vrow = &Vs2[buf + tl][d * PF_VLD + (g / 2) * 16 + (g % 2) * 4];
        *(uint2*)vrow = make_uint2(rv[i].x, rv[i].y);
        *(uint2*)(vrow + 8) = make_uint2(rv[i].z, rv[i].w);
      }
    }
  };
  auto stash = [&](const uint4* rk, const uint4* rv, int buf) {
    stash_k(rk, buf);
    stash_v(rv, buf);
  };
  const int kt0 = (b_lo / (RT * PF_BK)) * (RT * PF_BK);
  // The scores of one tile, out of LDS buffer `buf`: S^T = K . Q^T.
  auto scores = [&](int buf, floatx16 (&sc)[2]) {
    const bf16_t* Ks = Ks2[buf];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[ks][r] = 0.f;
#pragma unroll
      for (int kd = 0; kd < D16; ++kd) {
        const bf16x8_t kf = __builtin_bit_cast(bf16x8_t, *(const uint4*)&Ks[(ks * 32 + col) * KLD + kd * 16 + hf * 8]);
        sc[ks] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kd], sc[ks], 0, 0, 0);
      }
    }
  };
  // Mask, running maximum, weights, and the weighted sum of the tile's values out of LDS buffer `buf`.
  // WHOLE: every row of the wavefront sees all of the tile's keys, known when compiled (no mask, no branch).
  auto weigh = [&](int kt, int buf, floatx16 (&sc)[2], auto wholec) {
    constexpr bool WHOLE = decltype(wholec)::value;
    const bf16_t* Vs = Vs2[buf];
    {
      // Mask, running maximum and weights.  The maximum is kept in the base-2 domain
      // (s * scale * log2 e, scale > 0), so that a weight costs one multiply-add and one hardware
      // exp2.  A tile that every row of the wavefront sees whole needs no mask at all; elsewhere a key
      // outside q_lo .. pq gets -inf added (0 otherwise), computed from the sign of
      // min(pq - key, key - q_lo) without a comparison: scores are finite, keys that do not exist
      // were loaded as zeros.
      const bool whole = WHOLE || (kt + PF_BK - 1 <= w_first && (window <= 0 || kt >= w_last - window + 1));
      float tmax = -INFINITY;
#ifdef PF_REL
      // Scores go to the base-2 domain here, with the row's scale and the bias of each key's distance.
      const int d0 = (q_ok ? pq : -(1 << 30)) - kt - 4 * hf;      // pq - key for the lane's first key
      const int e0 = (pq - q_lo) - d0;                             // key - q_lo likewise
      const bool far = kt + PF_BK - 1 <= w_first - (n_rel - 1);    // every key n_rel - 1 or more behind every row
      const float bfar = brel[0];
      // the lane's key c of the tile lies d0 - c behind its row: place (rel_len - 1 - PF_REL_PAD - d0) + c.  One
      // clamp a tile keeps rows that do not exist inside the table; rows that do never reach it (see PF_REL_PAD).
      const int d0c = d0 < 59 - PF_REL_PAD ? 59 - PF_REL_PAD : (d0 > n_rel - 1 + PF_REL_PAD ? n_rel - 1 + PF_REL_PAD : d0);
      const float* bp = brel + (rel_len - 1 - PF_REL_PAD - d0c);
      // three straight-line forms, chosen by conditions that hold for the whole wavefront
      if (whole && far) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float v = __builtin_fmaf(sc[ks][r], scale2, bfar);
            sc[ks][r] = v;
            tmax = fmaxf(tmax, v);
          }
      } else if (whole) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float v = __builtin_fmaf(sc[ks][r], scale2, bp[ks * 32 + 8 * (r / 4) + (r % 4)]);
            sc[ks][r] = v;
            tmax = fmaxf(tmax, v);
          }
      } else {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int c = ks * 32 + 8 * (r / 4) + (r % 4);
            const int lo = min(d0 - c, e0 + c);
            const float v = __builtin_fmaf(sc[ks][r], scale2, bp[c]) + __builtin_bit_cast(float, (lo >> 31) & (int)0xff800000);
            sc[ks][r] = v;
            tmax = fmaxf(tmax, v);
          }
      }
#else
      if (whole) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sc[ks][r]);
      } else {
        const int d0 = (q_ok ? pq : -(1 << 30)) - kt - 4 * hf;      // pq - key for the lane's first key
        const int e0 = (pq - q_lo) - d0;                             // key - q_lo likewise
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int c = ks * 32 + 8 * (r / 4) + (r % 4);
            const int lo = min(d0 - c, e0 + c);
            const float bias = __builtin_bit_cast(float, (lo >> 31) & (int)0xff800000);
            const float v = sc[ks][r] + bias;
            sc[ks][r] = v;
            tmax = fmaxf(tmax, v);
          }
      }
#endif
#ifdef PF_REL
      tmax = half_max(tmax);                           // over both halves of the wavefront: all 64 keys of the row
#else
      tmax = half_max(tmax) * scale2;                  // over both halves of the wavefront: all 64 keys of the row
#endif
      const float m_new = fmaxf(m, tmax);
      const bool any = m_new != -INFINITY;             // a row that has seen no key yet keeps zeros
      const float m_use = any ? m_new : 0.f;           // -inf - 0 stays -inf: weight 0, never NaN
      const float alpha = __builtin_amdgcn_exp2f(m - m_use);
      float tsum = 0.f;
      bf16x8_t pf[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          uint32_t u[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
#ifdef PF_REL
            const float p0 = __builtin_amdgcn_exp2f(sc[ks][kb * 8 + 2 * e] - m_use);
            const float p1 = __builtin_amdgcn_exp2f(sc[ks][kb * 8 + 2 * e + 1] - m_use);
#else
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[ks][kb * 8 + 2 * e], scale2, -m_use));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[ks][kb * 8 + 2 * e + 1], scale2, -m_use));
#endif
            tsum += p0 + p1;
            u[e] = pack2_bf16(p0, p1);
          }
          pf[ks][kb] = __builtin_bit_cast(bf16x8_t, make_uint4(u[0], u[1], u[2], u[3]));
        }
      l = l * alpha + tsum;                            // this half's keys only: the halves' sums meet at the end
      m = m_new;
      // (skipping this when no row's maximum rose was measured: no gain, some row of 32 mostly has a new one)
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc_o[i][r] *= alpha;
      // O^T += V^T . P^T ; the lane's 8 keys of a 16-key block are 4hf..4hf+3 and 8+4hf..8+4hf+3, which
      // lie side by side in the parked tile
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) {
            const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, *(const uint4*)&Vs[(i * 32 + col) * PF_VLD + ks * 32 + kb * 16 + 8 * hf]);
            acc_o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[ks][kb], acc_o[i], 0, 0, 0);
          }
    }
  };
  // the products of one tile, out of LDS buffer `buf`
  auto tile = [&](int kt, int buf) {
    if (wave_on && kt <= w_last && kt + PF_BK - 1 >= w_lo) {
      floatx16 sc[2];
      scores(buf, sc);
      weigh(kt, buf, sc, std::false_type{});
    }
  };

  // Steady state, two tiles a round, without a branch around the loads: the compiler then counts the
  // loads in flight exactly and a tile waits for its own registers only.  It lasts while the tile
  // asked for (two ahead) lies whole inside the workgroup's keys; the last tiles run through the
  // same steps with conditions and the clamping loads.  One barrier a tile: the buffer written now
  // was last read two tiles ago, before the previous barrier.
  if constexpr (KP == 1) {
  int kt = kt0;
  // Where the keys start at a tile's edge (no window, or one that happens to) and the steady state runs
  // at least once, its first two tiles are asked for the way it asks for all others: the loop is then
  // entered with the same loads in flight, in the same order, as it is re-entered, and the compiler counts
  // exactly how many may stay in flight at each wait.  (Entered after the clamping loads it waited for all
  // of them, and every second tile's keys had one tile's time to arrive instead of two.)  Elsewhere the
  // loop below, which takes any tile, does all of them.
  if (b_lo == kt0 && kt0 + 4 * PF_BK - 1 <= b_last) {
    fetch_fast(rk0, rv0, kt0);
    if (Q_LATE) load_q();
    fetch_fast(rk1, rv1, kt0 + PF_BK);
    for (; kt + 4 * PF_BK - 1 <= b_last; kt += 2 * PF_BK) {
      stash(rk0, rv0, 0);
      lds_barrier();
      fetch_fast(rk0, rv0, kt + 2 * PF_BK);
      tile(kt, 0);
      stash(rk1, rv1, 1);
      lds_barrier();
      fetch_fast(rk1, rv1, kt + 3 * PF_BK);
      tile(kt + PF_BK, 1);
    }
  } else {
    fetch(rk0, rv0, kt0);
    if (Q_LATE) load_q();
    if (kt0 + PF_BK <= b_last) fetch(rk1, rv1, kt0 + PF_BK);
  }
  for (int parity = 0; kt <= b_last; kt += PF_BK, parity ^= 1) {
    if (parity == 0) {
      stash(rk0, rv0, 0);
      lds_barrier();
      if (kt + 2 * PF_BK <= b_last) fetch(rk0, rv0, kt + 2 * PF_BK);
    } else {
      stash(rk1, rv1, 1);
      lds_barrier();
      if (kt + 2 * PF_BK <= b_last) fetch(rk1, rv1, kt + 2 * PF_BK);
    }
    tile(kt, parity);
  }
  } else {
    // Key phases: a round parks KP tiles (one register set: the next round's loads fly while this
    // round's tiles are multiplied), each wavefront multiplies the tile of its phase.  Two barriers a
    // round: the tiles are parked before anyone reads them and read before they are replaced.
    if (b_lo == kt0 && kt0 + KP * PF_BK - 1 <= b_last) fetch_fast(rk0, rv0, kt0);     // (a first round that is whole: no clamping)
    else fetch(rk0, rv0, kt0);
    for (int kt = kt0; kt <= b_last; kt += KP * PF_BK) {
      stash(rk0, rv0, 0);
      lds_barrier();
      const int nx = kt + KP * PF_BK;
      if (nx + KP * PF_BK - 1 <= b_last) fetch_fast(rk0, rv0, nx);     // (nx >= b_lo: only the first round starts below it)
      else if (nx <= b_last) fetch(rk0, rv0, nx);
      tile(kt + kp * PF_BK, kp);
      lds_barrier();
    }
    // the phases' partial results, merged by phase 0 in the order of the phases
    l += __shfl_xor(l, 32, DA_WAVE);                    // (both halves had the same maximum all along)
    float* mg = (float*)smem;
    constexpr int PER = DT * 16 + 2;
    if (kp > 0) {
      float* mine = mg + (size_t)((kp - 1) * RB + rbi) * PER * DA_WAVE + lane;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(i * 16 + r) * DA_WAVE] = acc_o[i][r];
      mine[(DT * 16) * DA_WAVE] = m;
      mine[(DT * 16 + 1) * DA_WAVE] = l;
    }
    lds_barrier();
    if (kp > 0) return;
#pragma unroll
    for (int k = 1; k < KP; ++k) {
      const float* theirs = mg + (size_t)((k - 1) * RB + rbi) * PER * DA_WAVE + lane;
      const float mk = theirs[(DT * 16) * DA_WAVE], lk = theirs[(DT * 16 + 1) * DA_WAVE];
      const float m_new = fmaxf(m, mk);
      const float m_use = m_new != -INFINITY ? m_new : 0.f;
      const float a0 = __builtin_amdgcn_exp2f(m - m_use), a1 = __builtin_amdgcn_exp2f(mk - m_use);
      l = l * a0 + lk * a1;
      m = m_new;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc_o[i][r] = acc_o[i][r] * a0 + theirs[(i * 16 + r) * DA_WAVE] * a1;
    }
  }

  if constexpr (KP == 1) l += __shfl_xor(l, 32, DA_WAVE);   // (both halves had the same maximum all along)
  if (q_ok) {
    const float inv = 1.0f / l;
    bf16_t* orow = out + (size_t)(row0 + qi) * out_ld + h * D;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int d = i * 32 + 8 * r4 + 4 * hf;
        if (d < D) {
          const uint32_t lo2 = pack2_bf16(acc_o[i][r4 * 4] * inv, acc_o[i][r4 * 4 + 1] * inv);
          const uint32_t hi2 = pack2_bf16(acc_o[i][r4 * 4 + 2] * inv, acc_o[i][r4 * 4 + 3] * inv);
          *(uint2*)(orow + d) = make_uint2(lo2, hi2);
        }
      }
  }
}

#ifndef DA_ATTN_BODIES
// Whether q is asked for behind the first tile's keys and values: a row a lane is the slow way through a compute unit's address unit (64 cycles a load), and
// in front of the block table's entries everything waits for it.  But its registers are then held beside the tiles': at head sizes of 48 and 64 the form
// without phases loses the third workgroup that its LDS has room for, with a bias at 80 the second, and head sizes above 200 spill.  us, in front / behind, head
// size 64 without phases, prompts of 1,024: 2 x 25 heads (400 workgroups) 24.8 / 23.5, 5 x 16 (640) 26.4 / 24.9, 6 x 16 (768) 28.5 / 30.3, 8 x 12 (768)
// 28.2 / 30.9, 8 x 25 (1,600) 55.0 / 60.1; 16 x 512, 12 heads (768) 19.1 / 20.9; few long ones, whose first workgroups walk alone at the end: 6,000 x 16 (752) 124 / 110,
// 8,192 x 12 (768) 161 / 149, but 8,192 x 25 (1,600) 311 / 323.  With a bias 8 x 1,024 x 16 at 64 43.3 / 41.4, at 112 94.2 / 88.4, at 128 95.4 / 89.1, at 80
// 53.4 / 67.5, at 96 level.  Forms with phases: 1,024 x 12 17.2 / 17.8, 4 x 64 rows after 900 keys 15.8 / 17.6, 8 x 16 after 1,000 20.9 / 21.7, head size 48
// 2 x 1,024 x 16 16.8 / 18.9.  Other head sizes level or behind: 160 37.6 / 38.7, 240 57.3 / 62.4, 256 65.4 / 76.8.
#ifdef PF_REL
static constexpr bool pf_q_late(int D) { return D == 64 || D == 112 || D == 128; }
#define PF_LAUNCH_41(N) LAUNCH3(N, 4, 1, pf_q_late(16 * N))
#else
static bool pf_q_late(int D, long workgroups, int max_query_len) { return D == 64 && workgroups <= (max_query_len >= 4096 ? 800 : 640); }
#define PF_LAUNCH_41(N)                                                        \
  do {                                                                         \
    if (N == 4 && pf_q_late(16 * N, per128, max_query_len)) LAUNCH3(N, 4, 1, (N == 4)); \
    else LAUNCH3(N, 4, 1, false);                                              \
  } while (0)
#endif

#ifdef PF_REL
extern "C" int da_attn_prefill_rel_max_dist() { return PF_REL_MAX_DIST; }

extern "C" int da_attn_prefill_rel(const void* q, int q_ld, const void* cache, const int* block_table,
                                   int max_blocks, const int* q_start, const int* seq_lens, int seq0, int n_seqs,
                                   int max_query_len, int Hq, int Hkv, int D, int page, float scale, int window,
                                   const float* rel_bias, int n_dist, float t_coef, int t_every,
                                   void* out, int out_ld, int form, void* stream) {
  DA_REQUIRE(!rel_bias || (n_dist > 0 && n_dist <= PF_REL_MAX_DIST), "attn_prefill_rel: a bias table of %d entries (1 to %d are taken)",
             n_dist, PF_REL_MAX_DIST);
  DA_REQUIRE(t_every >= 0, "attn_prefill_rel: bad temperature period %d", t_every);
  DA_REQUIRE(D <= 128, "attn_prefill_rel: head size %d (up to 128 is taken)", D);
#else
extern "C" int da_attn_prefill(const void* q, int q_ld, const void* cache, const int* block_table,
                               int max_blocks, const int* q_start, const int* seq_lens, int seq0, int n_seqs,
                               int max_query_len, int Hq, int Hkv, int D, int page, float scale, int window,
                               void* out, int out_ld, int form, void* stream) {
#endif
  DA_REQUIRE(n_seqs >= 0 && Hq > 0 && Hkv > 0 && page > 0 && max_query_len >= 0, "attn_prefill: bad sizes");
  DA_REQUIRE(Hq % Hkv == 0, "attn_prefill: %d query heads are not a multiple of %d key heads", Hq, Hkv);
  DA_REQUIRE(D % 16 == 0 && D >= 16 && D <= 256, "attn_prefill: head size %d is not a multiple of 16 up to 256", D);
  DA_REQUIRE(page >= 8 && (page & (page - 1)) == 0 && PF_BK % page == 0, "attn_prefill: page size %d must be 8, 16, 32 or 64", page);
  DA_REQUIRE(q_ld >= Hq * D && out_ld >= Hq * D && q_ld % 8 == 0 && out_ld % 4 == 0, "attn_prefill: row lengths");
  DA_REQUIRE(((uintptr_t)q % 16 == 0) && ((uintptr_t)cache % 16 == 0) && ((uintptr_t)out % 8 == 0),
             "attn_prefill: operands must be 16-byte aligned");
  DA_REQUIRE(window >= 0 && max_blocks > 0, "attn_prefill: bad window or block table");
  DA_REQUIRE(scale > 0.f, "attn_prefill: the score scale must be positive, found %g", (double)scale);
  DA_REQUIRE((long)n_seqs * Hq < (1L << 31) && max_query_len <= 65535 * 32, "attn_prefill: too many sequences, heads or rows for one launch");
  if (n_seqs == 0 || max_query_len == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  // The workgroup's form, row blocks x key phases.  Short portions (after a long past, beside decoded
  // tokens) have few rows to a sequence and head: 1 x 4 up to 32 rows, 2 x 2 up to 64, so that all four
  // wavefronts work and share out the keys (see below for how many keys).  Longer ones take 128 rows a workgroup (smaller row blocks
  // read the keys more often, and that traffic binds), and 4 x 2, eight wavefronts, while there is no
  // more than one workgroup a compute unit; else 4 x 1.  Measured on MI355X, head size 64, microseconds
  // 4x1 / 4x2 / 2x2 / 1x4: 4 x 64 rows after 900 keys 19.8 / 17.0 / 15.6 / 19.3; 16 x 2 rows after 1,000 keys 20.2 / 17.6 / 16.7 / 24.2 (one
  // sequence of 8 or 64 rows: below).  4x1 / 4x2: 2 x 1,024 rows, 12 heads 19.6 / 17.9, 25 heads 23.5 / 23.4; 2,048 rows 33.0 / 29.3; 8 x 512 rows
  // 14.0 / 15.9; 8 x 1,024 rows, 12 heads 28.5 / 35.2 (452 TFLOP/s), 25 heads 54.5 / 69.8 (493); 2 x 4,096 rows 79.9 / 92.5 (645); 8,192 rows
  // 145.5 / 171.2 (709); 4 x 512 rows after 512 keys, 16 heads 19.2 / 17.9.  Workgroups of 256 rows (8 x 1) were behind 4 x 1 at every one of these.  A loop that multiplies
  // the scores of tile j + 1 while tile j is weighed (keys parked one tile ahead of values) gave the same bits and
  // -8 % to +12 % of 4 x 1's time depending on the shape: with two wavefronts a SIMD the matrix cores already run under
  // the other wavefront's softmax; it is not kept.  Four key phases (2 x 4, 4 x 4) were behind 4 x 2 at every shape (2 x
  // 1,024 rows, 12 heads: 20.5 and 22.3 against 18.3 us): a round's two barriers and the merge cost more than they share out.
  // Forms with phases need their tiles in LDS at once: head sizes up to 64 (4 x 2, 1 x 4) or 128 (2 x 2).  The
  // choice reads the step's shape only.
  // form: 0 leaves the choice to this rule; 41, 42, 22 or 14 fixes it
  const long per128 = (long)da_ceil_div(max_query_len, 128) * Hq * n_seqs;
  // Up to 64 rows, by the most keys that any sequence has (the block table's width), head size 64, us 4x1 / 2x2 / 1x4, 12 heads, 8 and 64
  // rows: 64 keys 4.5 / 6.0 / 9.3 and 4.9 / 6.5 / 10.0 (one tile: there is nothing to share out, and a round that is not whole
  // asks for its tiles the slow way); 128 keys 5.9 / 5.0 / 8.9 and 6.2 / 5.4 / 9.6; 256 7.2 / 6.1 / 6.9 and 7.6 / 6.6 / 9.0; 512 11.0 / 8.4 / 8.7 and
  // 11.4 / 8.9 / 12.3; 1,024 18.8 / 13.0 / 12.3 and 19.2 / 13.6 / 16.0.  So 4 x 1 up to one tile, 1 x 4 for up to 32 rows with
  // more than 768 keys, else 2 x 2.  Head sizes up to 32, with half the work a tile or less: 1 x 4 from more than 384 keys on (head size
  // 32, 2x2 / 1x4: 320 keys 6.8 / 7.6, 448 7.6 / 7.3, 640 7.8 / 8.5, 704 9.2 / 8.4, 1,024 10.1 / 8.5; 16: 448 7.3 / 6.8; 48: as 64).
  const long keys = (long)max_blocks * page;
#ifdef PF_REL
  const bool one_tile = false, far = true;          // (measured without a bias only)
#else
  const bool one_tile = D <= 64 && keys <= PF_BK, far = keys > (D <= 32 ? 384 : 768);
#endif
  const int chosen = form ? form
                     : (one_tile && max_query_len <= 64) ? 41
                     : (D <= 64 && max_query_len <= 32 && far) ? 14
                     : (D <= 128 && max_query_len <= 64) ? 22
                     : (D <= 64 && per128 <= PF_PHASED_MAX_WORKGROUPS) ? 42 : 41;
  DA_REQUIRE(chosen == 41 || (chosen == 22 && D <= 128) || ((chosen == 42 || chosen == 14) && D <= 64),
             "attn_prefill: form %d with a head size of %d (41 for any; 22 up to 128; 42 and 14 up to 64)", chosen, D);
  // every key a workgroup can see lies within max_blocks pages
  const bool bt_lds = max_blocks <= (chosen == 41 ? PF_BT_MAX : PF_BT_MAX_PHASED);
#define LAUNCH2(N, RB, KP, L, Q)                                                                               \
  hipLaunchKernelGGL((PF_KERNEL<N, RB, KP, L, Q>), dim3(Hq, n_here, da_ceil_div(max_query_len, 32 * RB)), \
                     dim3(RB * KP * DA_WAVE), 0, st, (const bf16_t*)q, (const bf16_t*)cache, block_table, q_start, seq_lens, \
                     q_ld, max_blocks, Hq, Hkv, s0, page, scale, window, (bf16_t*)out, out_ld PF_REL_ARGS)
#define LAUNCH3(N, RB, KP, Q)                \
  do {                                       \
    if (bt_lds) LAUNCH2(N, RB, KP, true, Q); \
    else LAUNCH2(N, RB, KP, false, Q);       \
  } while (0)
#define LAUNCH_SMALL(N)                            \
  case N:                                          \
    if (chosen == 14) LAUNCH3(N, 1, 4, false);     \
    else if (chosen == 22) LAUNCH3(N, 2, 2, false); \
    else if (chosen == 42) LAUNCH3(N, 4, 2, false); \
    else PF_LAUNCH_41(N);                          \
    break;
#define LAUNCH_MID(N)                              \
  case N:                                          \
    if (chosen == 22) LAUNCH3(N, 2, 2, false);     \
    else PF_LAUNCH_41(N);                          \
    break;
#define LAUNCH(N)                                  \
  case N:                                          \
    PF_LAUNCH_41(N);                               \
    break;
  // (a head, a sequence and a row block a workgroup, found without a division; a launch's second size ends at 65,535)
  for (int s0 = seq0; s0 < seq0 + n_seqs; s0 += 65535) {
    const int n_here = seq0 + n_seqs - s0 < 65535 ? seq0 + n_seqs - s0 : 65535;
    switch (D / 16) {
      LAUNCH_SMALL(1) LAUNCH_SMALL(2) LAUNCH_SMALL(3) LAUNCH_SMALL(4) LAUNCH_MID(5) LAUNCH_MID(6) LAUNCH_MID(7) LAUNCH_MID(8)
#ifndef PF_REL
      LAUNCH(9) LAUNCH(10) LAUNCH(11) LAUNCH(12) LAUNCH(13) LAUNCH(14) LAUNCH(15) LAUNCH(16)
#endif
    }
  }
#undef LAUNCH
#undef LAUNCH_MID
#undef LAUNCH_SMALL
#undef PF_LAUNCH_41
#undef LAUNCH3
#undef LAUNCH2
  DA_CHECK_LAUNCH("attn_prefill");
  return 0;
}
#endif
