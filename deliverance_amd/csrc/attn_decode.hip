// Paged attention for decode rows in bfloat16: one query row per sequence.
//
// One workgroup of 8 or 16 wavefronts per (sequence, query head).  The keys lo..p of the sequence
// are walked in aligned chunks of 64; wavefront v takes chunks v, v + 8 (16), ...  All loads of a chunk are
// issued before any is used, so a chunk costs two memory round trips: the block table's entries, then keys
// and values.  The arithmetic is on the matrix cores (MFMA 16x16x32), with one useful column in the first
// product and three in the second: a single wavefront's chain of instructions, not the chip's rate, is what a
// step of few requests waits for, and a chunk takes 16 instructions of 16 cycles here where it took about 700
// of the vector unit (one head of 64, 512 keys: 6.0 -> 5.7 us a launch in a recorded chain, of which 1.6 are
// the launch and about 2 the 130 KB that one compute unit pulls in; 64 sequences of 25 heads: 42.5 -> 40.7 us, 5.15 TB/s).
//   scores : 4 pieces of 16 keys, 16 bytes of a key's row a lane.  Four lanes that follow each other read 64 consecutive
//            bytes: a compute unit takes four lanes' addresses at once where they lie in one line, one at a time else (130 KB
//            alone: 2.5 against 4.8 us; a recorded step of 33 requests of the 355M's sizes 1,190 -> 1,153 us).  So row 4 a + b of the left operand holds, in k-group g, dimensions
//            8 b .. 8 b + 7 (of 32) of key g of the rows' group a, and column 4 g + b of the right operand is q's dimensions 8 b ..
//            in k-group g and zero elsewhere: the result's row 4 a + b, column 4 g + b is that key's share from these
//            dimensions, and four neighbouring lanes add up its four shares.  (Zero times an infinite key of the
//            same rows is no number: a chunk where one appears has its scores once more, a key a row.)  Products of
//            bfloat16 are exact and their sums 32-bit; the scale comes after.  us, a key a row / this, pages of 16: head size 64, 1 sequence of 12 heads
//            and 512 keys 5.4 / 4.5, 64 of 25 heads 35.3 / 35.1; with a bias, 640 keys, 5 of 16 heads 8.3 / 7.1, 64 of 16 31.7 / 31.4; head size 32, 64
//            sequences of 16 heads and 512 keys 13.8 / 13.8; 80, 32 of 600 21.8 / 22.0; 128, 4 of 600 10.0 / 7.6; 256, 32 of 8 heads 32.2 / 32.5, with a
//            bias 38.2 / 34.4; behind at 48 (64 of 600 22.7 / 23.1) and 16 (8 of 8 heads 4.1 / 4.3; 64 of 16 10.6 / 10.3).
//   softmax: four neighbouring lanes hold the same 4 keys that follow each other.  Running maximum and sum per wavefront
//            (the recurrence of native/src/main/resources/decode_paged_attention_f32.wgsl:31-65).
//   values : O[d, part] += V^T[d, key] . P[key, part]; values are stored dimension-major, so the left operand is
//            16 bytes as they lie in the page.  The 32-bit weights lose nothing: column 0 takes a weight rounded to
//            bfloat16, column 1 what is left rounded again, column 2 what is left of that (3 x 8 bits hold a 32-bit
//            number's 24), and the three columns' sums are added at the end.
// The wavefronts' partial results are merged in LDS in a fixed order.  Every sum's order
// depends on p and lo only, never on the batch.
//
// Formulas: core/src/main/java/io/teknek/deliverance/generator/CausalSelfAttention.java:504-532;
// tensor/src/main/java/io/teknek/deliverance/tensor/operations/TensorOperations.java:240-272.
//
// Compiled a second time with DEC_REL (attn_decode_rel.hip) the kernel also takes what some designs put on the
// scores: a bias by the distance between query and key (a table [Hq][n_dist], 32-bit, the last entry for every
// larger distance) and a query temperature 1 + t_coef * ln(floor((p + 1) / t_every) + 1) that multiplies the
// scale; a slope per head that a score loses for every position of distance; chunks of positions in place of a window (a row sees the keys of its own chunk only); a sink, one number a head
// whose exponential joins the softmax's denominator, without a key or a value and not scaled; and a gate, rows like out,
// of which o is multiplied with the logistic function.  The last two act once, after everything has been merged.  The
// plain build has none of that code.
#include "gemm_common.h"
#include <da_anew.h>
#include <da_read_arg.h>

#define DEC_MAX_D 256

#ifdef DEC_REL
#define DEC_KERNEL attn_decode_rel_kernel
#define DEC_MERGE_KERNEL attn_decode_rel_merge_kernel
#define DEC_REL_PARAMS , const float* __restrict__ rel_bias, int n_dist, const float* __restrict__ slopes, float t_coef, int t_every, int chunk DEC_END_PARAMS
#define DEC_REL_DECL , const float* rel_bias, int n_dist, const float* slopes, float t_coef, int t_every, int chunk, const float* sink, const bf16_t* gate, int gate_ld
#define DEC_REL_ARGS , rel_bias, n_dist, slopes, t_coef, t_every, chunk DEC_END_ARGS
#define DEC_END_PARAMS , const float* __restrict__ sink, const bf16_t* __restrict__ gate, int gate_ld
#define DEC_END_ARGS , sink, gate, gate_ld
#define DEC_REL_OF_ROWS(s0) , rel_bias, n_dist, slopes, t_coef, t_every, chunk, sink, gate ? gate + (size_t)(s0) * gate_ld : nullptr, gate_ld
#else
#define DEC_KERNEL attn_decode_kernel
#define DEC_MERGE_KERNEL attn_decode_merge_kernel
#define DEC_REL_PARAMS
#define DEC_REL_DECL
#define DEC_REL_ARGS
#define DEC_END_PARAMS
#define DEC_END_ARGS
#define DEC_REL_OF_ROWS(s0)
#endif

// e^x by the hardware's exp2 (two instructions; the library's expf is a dozen, and the merge of 16 wavefronts'
// partial results takes 16 of them on the one wavefront that everything waits for)
__device__ __forceinline__ float dec_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

#ifdef DEC_REL
// What a finished row is multiplied with, from its maximum and its sum of weights: one over the sum, which the sink
// joins; `shrink` is what its term makes of the weights' common scale.
__device__ __forceinline__ float dec_inverse(float mm, float ll, bool with_sink, float s0) {
  float shrink = 1.f;
  if (with_sink) {
    const float m_all = fmaxf(mm, s0);
    shrink = mm == -INFINITY ? 0.f : dec_exp(mm - m_all);
    ll = ll * shrink + dec_exp(s0 - m_all);
  }
  return ll > 0.f ? shrink / ll : 0.f;
}
// a number that is the same in all lanes, in a scalar register
__device__ __forceinline__ float dec_of_all(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}
__device__ __forceinline__ float dec_gate(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
#endif

// Long contexts with few (sequence, head) pairs: the keys are also split over workgroups.  Workgroup
// (pair, j) takes the keys j * span .. (j + 1) * span - 1 (span a multiple of 64) and leaves its
// partial result (the weighted sum before the division, the maximum, the sum of weights: D + 2
// floats) in a scratch buffer; a second kernel merges a pair's partial results in ascending order
// of j.  The split depends on the step's shape only (pairs, widest block table), never on the
// sequences' lengths, so a recorded graph can hold it.
//
// DK: dimensions in steps of 32, rounded up to a power of two (1, 2, 4, 8)
// Included by attn_both.hip (DA_ATTN_BODIES) the kernel is a function that is told which workgroup it is.  (A function in both
// files, called by a kernel, compiles to other code: one-token steps of the Virudra 1,101 -> 1,106 us.)
template <int DK, int DEC_WAVES, bool SPLIT>
#ifdef DA_ATTN_BODIES
__device__ __forceinline__ void
attn_decode_body(int s, int h,
#else
// (registers are held to 128 for head sizes up to 64, so that two workgroups share a compute unit)
__global__ void __launch_bounds__(DEC_WAVES * DA_WAVE, (DK <= 2 || DEC_WAVES == 16) ? 4 : 2)
DEC_KERNEL(
#endif
           const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, const int* __restrict__ block_table,
           const int* __restrict__ seq_lens, int q_ld, int max_blocks, int Hq, int Hkv, int D, int page, float scale,
           int window, bf16_t* __restrict__ out, int out_ld, int span, float* __restrict__ partial DEC_REL_PARAMS) {
#ifndef DA_ATTN_BODIES
  const int h = blockIdx.x, s = blockIdx.y;
#endif
  constexpr int DV = 2 * DK;                  // pieces of 16 value dimensions
  constexpr int DMAX = 32 * DK;
  __shared__ __attribute__((aligned(16))) bf16_t ps[DEC_WAVES][4][DA_WAVE];     // a chunk's weights in three parts; part 3: zeros
  __shared__ __attribute__((aligned(16))) float part_acc[DEC_WAVES][DMAX];
  __shared__ float part_m[DEC_WAVES], part_l[DEC_WAVES];

  const int hk = Hq == Hkv ? h : h / (Hq / Hkv);
  const int t = threadIdx.x, lane = t % DA_WAVE, wave = __builtin_amdgcn_readfirstlane(t / DA_WAVE);
  const int col = lane % 16, quad = lane / 16;
  const int kd = 8 * (col % 4);               // the dimensions (of 32) that the lane loads of a key
  const int ka = 16 * (col / 4) + 4 * quad;   // the first of the 4 keys of a chunk that it loads
  const int* bt = block_table + (size_t)s * max_blocks;
  // addressing by shifts: the page size is a power of two (checked on the host)
  const int lg = 31 - __builtin_clz(page), pmask = page - 1;
  const uint32_t page_bytes = 4u * (uint32_t)(Hkv * page * D);
  const char* kbase = (const char*)(cache + (long long)hk * page * D);
  const char* vbase = (const char*)(cache + (long long)(Hkv + hk) * page * D);

  // Asked for before the sequence's length is known, so that they travel beside it: the query and the
  // block-table entries of the chunk this wavefront starts with when nothing is cut off by a window
  // (keys wave*64 ..).  Entries past the sequence's pages are read (the table has max_blocks of them) and
  // never used.  A lane's dimensions past D (a head size that is no multiple of 32) meet zeros of q.
  uint4 qf[DK];
#pragma unroll
  for (int k = 0; k < DK; ++k) {
    const int d = 32 * k + kd;
    qf[k] = *(const uint4*)(q + (size_t)s * q_ld + h * D + (d < D ? d : 0));
  }
  const int split0 = SPLIT ? (int)blockIdx.z * span : 0;          // the first key of this workgroup's share
  const int c0_guess = split0 + wave * DA_WAVE;
  int btk0, btv0[2];                          // (pages hold whole groups of 4 keys)
  {
    const int pg = (c0_guess + ka) >> lg;
    btk0 = bt[pg < max_blocks ? pg : max_blocks - 1];
  }
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int pg = (c0_guess + 32 * g + 8 * quad) >> lg;
    btv0[g] = bt[pg < max_blocks ? pg : max_blocks - 1];
  }
#ifdef DEC_REL
  // asked for here, used at the end
  const int gd = t < D ? t : 0;
  const bf16_t graw = !SPLIT && gate ? gate[(size_t)s * gate_ld + h * D + gd] : (bf16_t)0;
  const float s0 = !SPLIT && sink ? sink[h] : 0.f;
#endif
  // the arguments behind the first 14 words, now: each line of them that is first asked for at its use is a wait of its own
  da_read_arg(scale);
  da_read_arg(window);
  da_read_arg(out);
  da_read_arg(out_ld);
#ifdef DEC_REL
  da_read_arg(rel_bias);
  da_read_arg(slopes);
  da_read_arg(t_every);
  da_read_arg(gate_ld);
#endif
  // the row's position is seq_lens[s] - 1; it sees the keys lo..p (of which this workgroup takes its share)
  const int p_row = seq_lens[s] - 1;
#ifdef DEC_REL
  const int lo_row = chunk > 0 ? (p_row > 0 ? p_row / chunk * chunk : 0)
                               : ((window > 0 && p_row - window + 1 > 0) ? p_row - window + 1 : 0);
#else
  const int lo_row = (window > 0 && p_row - window + 1 > 0) ? p_row - window + 1 : 0;
#endif
  const int p = SPLIT ? (p_row < split0 + span - 1 ? p_row : split0 + span - 1) : p_row;
  const int lo = SPLIT ? (lo_row > split0 ? lo_row : split0) : lo_row;
#ifdef DEC_REL
  const float* brow = rel_bias ? rel_bias + (size_t)h * n_dist : nullptr;
  const float slope = dec_of_all(slopes ? slopes[h] : 0.f);
  const float qscale = dec_of_all(t_every > 0 ? scale * (1.0f + t_coef * logf((float)((p_row + 1) / t_every + 1))) : scale);
#else
  const float qscale = scale;
#endif
#pragma unroll
  for (int k = 0; k < DK; ++k)
    if (32 * k + kd >= D || quad != col / 4) qf[k] = make_uint4(0, 0, 0, 0);

  floatx4 acc[DV];
#pragma unroll
  for (int i = 0; i < DV; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  for (int c0 = (lo / DA_WAVE) * DA_WAVE + wave * DA_WAVE; c0 <= p; c0 += DEC_WAVES * DA_WAVE) {
    const int first = c0 > lo ? c0 : lo;                 // valid keys of the chunk: first..last
    const int last = c0 + DA_WAVE - 1 < p ? c0 + DA_WAVE - 1 : p;
    auto is_seen = [&](int key) { return (uint32_t)(key - first) <= (uint32_t)(last - first); };      // (one comparison: two of them become a branch)
    // the pages of the chunk's keys and value groups: those asked for at the start, or read now
    int btk, btv[2], bt_safe;
    if (c0 == c0_guess && first == c0) {                 // the same for the whole wavefront
      btk = btk0;
      btv[0] = btv0[0];
      btv[1] = btv0[1];
      bt_safe = __builtin_amdgcn_readfirstlane(btk0);    // lane 0 holds the page of key c0
    } else {
      bt_safe = bt[first >> lg];
      btk = bt[((c0 + ka + 3 >= first && c0 + ka <= last) ? c0 + ka : first) >> lg];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int g0 = c0 + 32 * g + 8 * quad;
        btv[g] = bt[((g0 + 7 >= first && g0 <= last) ? g0 : first) >> lg];
      }
    }
    // ---- all loads of the chunk, then the arithmetic.  A key that is not seen reads `first` instead, a row that
    // surely exists; of the values, a group of 8 keys (which never crosses a page) without a seen key reads the group
    // of `first` instead.  Both are dropped.
    // (head sizes above 128 have no registers for all of it: two pieces of keys at a time, the values once the scores
    // are done, half of the chunk at a time)
    constexpr bool EARLY_V = DK <= 4;
    constexpr int KJ = EARLY_V ? 4 : 2, VG = EARLY_V ? 2 : 1;
    uint4 kf[KJ][DK], vf[VG][DV];
    floatx4 sc[4];
    auto load_k = [&](int j0) {
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        const int key = c0 + ka + j0 + j;
        const bool valid = is_seen(key);
        const char* kp = kbase + (uint64_t)(uint32_t)(valid ? btk : bt_safe) * page_bytes +
                         (uint32_t)(2 * (((valid ? key : first) & pmask) * D + (DK > 1 || kd < D ? kd : D - 8)));
#pragma unroll
        for (int k = 0; k < DK; ++k)         // (D > 16 DK: only the upper half of the steps can lie past D; there the row's last piece is read, in its neighbours' line)
          kf[j][k] = *(const uint4*)(kp + (DK == 1 || 2 * k + 1 < DK || 32 * k + kd < D ? 64 * k : 2 * (D - 8 - kd)));
      }
    };
    // Zeros in place of what lanes past D read: q is zero there, but zero times an infinite key is no number.
    auto clear_k = [&]() {
#pragma unroll
      for (int k = DK / 2; k < DK; ++k) {
        const uint32_t keep = 32 * k + kd < D ? 0xffffffffu : 0u;
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          kf[j][k].x &= keep;
          kf[j][k].y &= keep;
          kf[j][k].z &= keep;
          kf[j][k].w &= keep;
        }
      }
    };
    auto scores = [&](int j0) {
      if (D < DMAX) clear_k();
#pragma unroll
      for (int j = 0; j < KJ; ++j) sc[j0 + j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < DK; ++k)
#pragma unroll
        for (int j = 0; j < KJ; ++j)
          sc[j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[j][k]), __builtin_bit_cast(bf16x8_t, qf[k]), sc[j0 + j], 0, 0, 0);
    };
    auto load_v = [&](int g0_) {
#pragma unroll
      for (int g = 0; g < VG; ++g) {
        const int g0 = c0 + 32 * (g0_ + g) + 8 * quad;
        const bool any = g0 + 7 >= first && g0 <= last;
        const int gs = any ? g0 : (first & ~7);
        const char* vp = vbase + (uint64_t)(uint32_t)(any ? btv[g0_ + g] : bt_safe) * page_bytes + (uint32_t)(2 * ((gs & pmask) + col * page));
#pragma unroll
        for (int i = 0; i < DV; ++i) {
          vf[g][i] = *(const uint4*)vp;
          vp += 16 * (i + 1) < D ? 32 * page : 0;        // (a whole piece past D reads the last one again and is dropped)
        }
      }
    };
#ifdef DEC_REL
    // the biases of the keys whose scores this lane will keep, asked for in front of the keys and values (a key past the
    // row's own position has no distance: it reads entry 0 and is dropped with its score)
    float brel[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int dist = p_row - (c0 + 16 * quad + 4 * (col / 4) + r);
      brel[r] = slopes ? -slope * (float)dist : 0.f;
      if (brow) brel[r] += brow[dist < 0 ? 0 : (dist < n_dist ? dist : n_dist - 1)];
    }
#endif
    load_k(0);
    if (EARLY_V) load_v(0);
    // nothing moves across this line: the compiler would otherwise push the value loads down behind
    // the scores to save registers, and a chunk would cost a third memory round trip
    __builtin_amdgcn_sched_barrier(0);
    scores(0);
    if (!EARLY_V) {
      load_k(EARLY_V ? 0 : 2);
      scores(EARLY_V ? 0 : 2);
    }
    // What a lane works out from its number from here on is worked out here.  Held in registers across the loads, where keys, values and results
    // fill them, it takes a compute unit's third workgroup at head sizes up to 32 (92 registers for 77; 64 sequences of 16 heads and 512 keys 14.7 us for
    // 13.8) and spills at 64 with a bias (34.1 for 31.4) and above 128 (36.7 for 32.5).
    const uint32_t ln = da_anew((uint32_t)lane), ln16 = ln % 16, ln_quad = ln / 16, part = ln % 4;
    // this lane's 4 keys: piece r's row group ln_quad, k-group ln16 / 4; lane b of four neighbouring ones has their share b in register b
    const int key0 = c0 + (int)(16 * ln_quad + ln16 / 4 * 4);
    float sv[4], e[4];
    auto finish = [&](int r) {
      sv[r] *= qscale;
#ifdef DEC_REL
      sv[r] += brel[r];
#endif
      sv[r] = is_seen(key0 + r) ? sv[r] : -INFINITY;
    };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // (every lane takes the four shares from their lanes: a lane that picked its own would do so by comparisons with each place)
      const float s01 = dpp_move<0x00, 0xF>(sc[r][0], sc[r][0]) + dpp_move<0x55, 0xF>(sc[r][1], sc[r][1]);
      const float s23 = dpp_move<0xAA, 0xF>(sc[r][2], sc[r][2]) + dpp_move<0xFF, 0xF>(sc[r][3], sc[r][3]);
      sv[r] = s01 + s23;
      finish(r);
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(sv[0] != sv[0] || sv[1] != sv[1] || sv[2] != sv[2] || sv[3] != sv[3]) != 0, 0)) {
      // the chunk's scores once more, a key a row of the left operand and q in all columns: product j holds this lane's keys if j = ln16 / 4
#pragma unroll 1
      for (int j = 0; j < 4; ++j) {
        const int key = c0 + (int)(16 * (ln16 / 4) + 4 * j + part), seen = is_seen(key) ? key : first;
        const char* kp = kbase + (uint64_t)(uint32_t)bt[seen >> lg] * page_bytes + (uint32_t)(2 * (seen & pmask) * D);
        floatx4 one = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int k = 0; k < DK; ++k) {
          const int d = 32 * k + 8 * (int)ln_quad;
          uint4 kx = make_uint4(0, 0, 0, 0), qx = kx;
          if (d < D) {
            kx = *(const uint4*)(kp + 2 * d);
            qx = *(const uint4*)(q + (size_t)s * q_ld + h * D + d);
          }
          one = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kx), __builtin_bit_cast(bf16x8_t, qx), one, 0, 0, 0);
        }
        if (j == (int)(ln16 / 4)) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            sv[r] = one[r];
            finish(r);
          }
        }
      }
    }
    const float m_new = fmaxf(m, wave_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]))));
    const float alpha = dec_exp(m - m_new);              // (a chunk that is walked has a seen key: m_new is finite)
#pragma unroll
    for (int r = 0; r < 4; ++r) e[r] = dec_exp(sv[r] - m_new);
    l = l * alpha + 0.25f * wave_sum((e[0] + e[1]) + (e[2] + e[3]));      // (four lanes hold each key)
    m = m_new;
    {
      // of four neighbouring lanes the first parks the first part of their 4 weights, the others the second, the third, zeros
      uint32_t w2[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float a = e[2 * i], b = e[2 * i + 1];
        const uint32_t p0 = pack2_bf16(a, b);
        const float a1 = a - __uint_as_float(p0 << 16), b1 = b - __uint_as_float(p0 & 0xffff0000u);
        const uint32_t p1 = pack2_bf16(a1, b1);
        const uint32_t p2 = pack2_bf16(a1 - __uint_as_float(p1 << 16), b1 - __uint_as_float(p1 & 0xffff0000u));
        w2[i] = part == 0 ? p0 : (part == 1 ? p1 : (part == 2 ? p2 : 0u));
      }
      *(uint2*)&ps[wave][part][16 * ln_quad + ln16 / 4 * 4] = make_uint2(w2[0], w2[1]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");   // LDS only: the value loads stay in flight
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
    for (int i = 0; i < DV; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][r] *= alpha;
    const bool cut = first != c0 || last != c0 + DA_WAVE - 1;         // the same for the whole wavefront
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      uint4 (&v)[DV] = vf[EARLY_V ? g : 0];
      if (!EARLY_V) {
        __builtin_amdgcn_sched_barrier(0);               // (not moved up among the scores: the keys' registers are free only now)
        load_v(EARLY_V ? 0 : g);
      }
      const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, *(const uint4*)&ps[wave][ln16 < 3 ? ln16 : 3][32 * g + 8 * ln_quad]);
      if (cut) {
        // Rows outside first..last were never written (or belong to someone else) and may hold anything:
        // their bits are cleared.  The seen rows of the lane's group are g0 + lo8 .. g0 + hi8.
        const int g0 = c0 + 32 * g + 8 * (int)ln_quad;
        const int lo8 = first - g0, hi8 = last - g0;
        uint32_t msk[4];
#pragma unroll
        for (int w = 0; w < 4; ++w)
          msk[w] = ((2 * w >= lo8 && 2 * w <= hi8) ? 0x0000ffffu : 0u) | ((2 * w + 1 >= lo8 && 2 * w + 1 <= hi8) ? 0xffff0000u : 0u);
#pragma unroll
        for (int i = 0; i < DV; ++i) {
          v[i].x &= msk[0];
          v[i].y &= msk[1];
          v[i].z &= msk[2];
          v[i].w &= msk[3];
        }
      }
#pragma unroll
      for (int i = 0; i < DV; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, v[i]), pf, acc[i], 0, 0, 0);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
  // a lane holds dimensions 16 i + 4 * quad + r of part col; parts 0..2 (and the zeros of column 3) are added.  (An
  // infinite value stays what the first part makes of it: the other parts may be zero or of the other sign.)
#pragma unroll
  for (int i = 0; i < DV; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float sum = group_sum<4>(acc[i][r]);
      acc[i][r] = fabsf(acc[i][r]) < INFINITY ? sum : acc[i][r];
    }
  if (col == 0) {
#pragma unroll
    for (int i = 0; i < DV; ++i) *(floatx4*)&part_acc[wave][16 * i + 4 * quad] = acc[i];
  }
  if (lane == 0) { part_m[wave] = m; part_l[wave] = l; }
  __syncthreads();
  // merge the wavefronts' partial softmaxes in a fixed order
#ifdef DEC_REL
  if (wave * DA_WAVE >= D) return;       // (a dimension a thread: without one, the sink's and the sum's exponentials are in the others' way)
#endif
  float mm = part_m[0];
#pragma unroll
  for (int w2 = 1; w2 < DEC_WAVES; ++w2) mm = fmaxf(mm, part_m[w2]);
  float ll = 0.f;
  float f[DEC_WAVES];
#pragma unroll
  for (int w2 = 0; w2 < DEC_WAVES; ++w2) {
    f[w2] = part_m[w2] == -INFINITY ? 0.f : dec_exp(part_m[w2] - mm);
    ll += part_l[w2] * f[w2];
  }
  if (SPLIT) {
    // the share's result before the division, its maximum and its sum of weights
    float* mine = partial + (((size_t)s * Hq + h) * gridDim.z + blockIdx.z) * (D + 2);
    for (int d = t; d < D; d += DEC_WAVES * DA_WAVE) {
      float o = 0.f;
#pragma unroll
      for (int w2 = 0; w2 < DEC_WAVES; ++w2) o += part_acc[w2][d] * f[w2];
      mine[d] = o;
    }
    if (t == 0) { mine[D] = mm; mine[D + 1] = ll; }
    return;
  }
#ifdef DEC_REL
  const float inv = dec_inverse(mm, ll, sink != nullptr, s0);
  if (t < D) {                                      // (a workgroup has at least 512 threads)
    float o = 0.f;
#pragma unroll
    for (int w2 = 0; w2 < DEC_WAVES; ++w2) o += part_acc[w2][t] * f[w2];
    o *= inv;
    if (gate) o *= dec_gate(bf16_to_f32(graw));
    out[(size_t)s * out_ld + h * D + t] = f32_to_bf16(o);
  }
#else
  const float inv = ll > 0.f ? 1.0f / ll : 0.f;     // a sequence of length 0 (padding) gives zeros
  for (int d = t; d < D; d += DEC_WAVES * DA_WAVE) {
    float o = 0.f;
#pragma unroll
    for (int w2 = 0; w2 < DEC_WAVES; ++w2) o += part_acc[w2][d] * f[w2];
    out[(size_t)s * out_ld + h * D + d] = f32_to_bf16(o * inv);
  }
#endif
}

#ifndef DA_ATTN_BODIES
// The partial results of a (sequence, head) pair, merged in ascending order of the shares.
__global__ void __launch_bounds__(256)
DEC_MERGE_KERNEL(const float* __restrict__ partial, int n_splits, int Hq, int D,
                         bf16_t* __restrict__ out, int out_ld DEC_END_PARAMS) {
  const int s = blockIdx.x / Hq, h = blockIdx.x % Hq;
  const float* mine = partial + (size_t)blockIdx.x * n_splits * (D + 2);
  float mm = -INFINITY;
  for (int j = 0; j < n_splits; ++j) mm = fmaxf(mm, mine[(size_t)j * (D + 2) + D]);
  float ll = 0.f;
  for (int j = 0; j < n_splits; ++j) {
    const float mj = mine[(size_t)j * (D + 2) + D];
    ll += mine[(size_t)j * (D + 2) + D + 1] * (mj == -INFINITY ? 0.f : dec_exp(mj - mm));
  }
#ifdef DEC_REL
  const float inv = dec_inverse(mm, ll, sink != nullptr, sink ? sink[h] : 0.f);
#else
  const float inv = ll > 0.f ? 1.0f / ll : 0.f;
#endif
  for (int d = threadIdx.x; d < D; d += blockDim.x) {
    float o = 0.f;
    for (int j = 0; j < n_splits; ++j) {
      const float mj = mine[(size_t)j * (D + 2) + D];
      o += mine[(size_t)j * (D + 2) + d] * (mj == -INFINITY ? 0.f : dec_exp(mj - mm));
    }
#ifdef DEC_REL
    if (gate) o *= dec_gate(bf16_to_f32(gate[(size_t)s * gate_ld + h * D + d]));
#endif
    out[(size_t)s * out_ld + h * D + d] = f32_to_bf16(o * inv);
  }
}

static int decode_checks(const void* q, int q_ld, const void* cache, int max_blocks, int S, int Hq, int Hkv, int D,
                         int page, int window, int out_ld) {
  DA_REQUIRE(S >= 0 && Hq > 0 && Hkv > 0 && page > 0, "attn_decode: bad sizes");
  DA_REQUIRE(Hq % Hkv == 0, "attn_decode: %d query heads are not a multiple of %d key heads", Hq, Hkv);
  DA_REQUIRE(D % 16 == 0 && D >= 16 && D <= DEC_MAX_D, "attn_decode: head size %d is not a multiple of 16 up to %d", D, DEC_MAX_D);
  DA_REQUIRE(page % 8 == 0 && DA_WAVE % page == 0, "attn_decode: page size %d must be 8, 16, 32 or 64", page);
  DA_REQUIRE(q_ld >= Hq * D && out_ld >= Hq * D, "attn_decode: row lengths too small");
  DA_REQUIRE(window >= 0 && max_blocks > 0, "attn_decode: bad window or block table");
  DA_REQUIRE((uintptr_t)cache % 16 == 0 && (uintptr_t)q % 16 == 0 && q_ld % 8 == 0,
             "attn_decode: q and the cache must be 16-byte aligned");
  return 0;
}

// n_splits == 1: one workgroup a (sequence, head) pair, no scratch.  n_splits > 1: the keys of a pair
// go to n_splits workgroups of `span` keys each, partial results through `partial`
// (S * Hq * n_splits * (D + 2) floats), then the merge kernel.
static int decode_launch(const void* q, int q_ld, const void* cache, const int* block_table, int max_blocks,
                         const int* seq_lens, int S, int Hq, int Hkv, int D, int page, float scale, int window,
                         void* out, int out_ld, int n_splits, int span, float* partial, hipStream_t st DEC_REL_DECL) {
  // (a head and a sequence a workgroup, found without a division; the second size of a launch ends at 65,535)
  constexpr int MAX_S = 65535;
  if (S > MAX_S) {
    const int part = da_ceil_div(S, da_ceil_div(S, MAX_S));
    for (int s0 = 0; s0 < S; s0 += part) {
      const int n = S - s0 < part ? S - s0 : part;
      decode_launch((const bf16_t*)q + (size_t)s0 * q_ld, q_ld, cache, block_table + (size_t)s0 * max_blocks, max_blocks, seq_lens + s0, n, Hq, Hkv,
                    D, page, scale, window, (bf16_t*)out + (size_t)s0 * out_ld, out_ld, n_splits, span,
                    partial ? partial + (size_t)s0 * Hq * n_splits * (D + 2) : nullptr, st DEC_REL_OF_ROWS(s0));
    }
    return 0;
  }
  // 8 wavefronts; 16 where the workgroups are no more than the compute units (a context above 512 is then
  // still one chunk a wavefront, and the larger workgroup's start is paid once per compute unit)
  const bool wide = (long)S * Hq * n_splits <= 256 && D <= 64;         // larger heads need the registers of 8 wavefronts
  dim3 grid(Hq, S, n_splits);
#define LAUNCH3(C, W, SP)                                                                                   \
  hipLaunchKernelGGL((DEC_KERNEL<C, W, SP>), grid, dim3(W * DA_WAVE), 0, st, (const bf16_t*)q, \
                     (const bf16_t*)cache, block_table, seq_lens, q_ld, max_blocks, Hq, Hkv, D, page, scale, window, \
                     (bf16_t*)out, out_ld, span, partial DEC_REL_ARGS)
#define LAUNCH2(C, W) do { if (n_splits > 1) LAUNCH3(C, W, true); else LAUNCH3(C, W, false); } while (0)
#define LAUNCH(C) do { if (wide) LAUNCH2(C, 16); else LAUNCH2(C, 8); } while (0)
  if (D <= 32) LAUNCH(1);
  else if (D <= 64) LAUNCH(2);
  else if (D <= 128) LAUNCH2(4, 8);
  else LAUNCH2(8, 8);
#undef LAUNCH
#undef LAUNCH2
#undef LAUNCH3
  if (n_splits > 1)
    hipLaunchKernelGGL(DEC_MERGE_KERNEL, dim3(S * Hq), dim3(D <= 64 ? 64 : (D <= 128 ? 128 : 256)), 0, st,
                       partial, n_splits, Hq, D, (bf16_t*)out, out_ld DEC_END_ARGS);
  return 0;
}

#ifdef DEC_REL
static int rel_checks(const float* rel_bias, int n_dist, int t_every) {
  DA_REQUIRE(!rel_bias || n_dist > 0, "attn_decode_rel: a bias table without entries");
  DA_REQUIRE(t_every >= 0, "attn_decode_rel: bad temperature period %d", t_every);
  return 0;
}

// n_splits <= 1: one workgroup a (sequence, head) pair; else the keys of a pair go to n_splits workgroups
// and `workspace` holds the partial results.
extern "C" int da_attn_decode_rel(const void* q, int q_ld, const void* cache, const int* block_table,
                                  int max_blocks, const int* seq_lens, int S, int Hq, int Hkv, int D, int page,
                                  float scale, int window, const float* rel_bias, int n_dist, const float* slopes,
                                  float t_coef, int t_every, int chunk, const float* sink, const void* gate, int gate_ld, void* out,
                                  int out_ld, int n_splits, void* workspace, long workspace_bytes, void* stream) {
  if (decode_checks(q, q_ld, cache, max_blocks, S, Hq, Hkv, D, page, window, out_ld)) return 1;
  if (rel_checks(rel_bias, n_dist, t_every)) return 1;
  DA_REQUIRE(chunk >= 0 && (chunk == 0 || window == 0), "attn_decode_rel: a window or chunks, not both");
  DA_REQUIRE(!gate || gate_ld >= Hq * D, "attn_decode_rel: the gate's rows are too short");
  int span = 0;
  if (n_splits > 1) {
    DA_REQUIRE(n_splits <= 64, "attn_decode_rel: %d shares (2 to 64 are taken)", n_splits);
    const long keys = (long)max_blocks * page;
    span = (int)(((keys + n_splits - 1) / n_splits + DA_WAVE - 1) / DA_WAVE * DA_WAVE);
    const long need = (long)S * Hq * n_splits * (D + 2) * (long)sizeof(float);
    DA_REQUIRE(workspace && (uintptr_t)workspace % 16 == 0 && workspace_bytes >= need,
               "attn_decode_rel: the workspace holds %ld bytes, %ld are needed", workspace_bytes, need);
  }
  if (S == 0) return 0;
  decode_launch(q, q_ld, cache, block_table, max_blocks, seq_lens, S, Hq, Hkv, D, page, scale, window, out, out_ld,
                n_splits > 1 ? n_splits : 1, span, (float*)workspace, (hipStream_t)stream, rel_bias, n_dist, slopes, t_coef, t_every,
                chunk, sink, (const bf16_t*)gate, gate_ld);
  DA_CHECK_LAUNCH("attn_decode_rel");
  return 0;
}
#else
extern "C" int da_attn_decode(const void* q, int q_ld, const void* cache, const int* block_table,
                              int max_blocks, const int* seq_lens, int S, int Hq, int Hkv, int D, int page,
                              float scale, int window, void* out, int out_ld, void* stream) {
  if (decode_checks(q, q_ld, cache, max_blocks, S, Hq, Hkv, D, page, window, out_ld)) return 1;
  if (S == 0) return 0;
  decode_launch(q, q_ld, cache, block_table, max_blocks, seq_lens, S, Hq, Hkv, D, page, scale, window, out, out_ld,
                1, 0, nullptr, (hipStream_t)stream);
  DA_CHECK_LAUNCH("attn_decode");
  return 0;
}

// The keys of every (sequence, head) pair split over n_splits workgroups; `workspace` holds the
// partial results (da_attn_decode_split_bytes of it, 16-byte aligned).
extern "C" long da_attn_decode_split_bytes(int S, int Hq, int D, int n_splits) {
  return (long)S * Hq * n_splits * (D + 2) * (long)sizeof(float);
}

static int split_checks(int max_blocks, int page, int n_splits, int* span) {
  DA_REQUIRE(n_splits >= 2 && n_splits <= 64, "attn_decode_split: %d shares (2 to 64 are taken)", n_splits);
  const long keys = (long)max_blocks * page;
  *span = (int)(((keys + n_splits - 1) / n_splits + DA_WAVE - 1) / DA_WAVE * DA_WAVE);
  return 0;
}

extern "C" int da_attn_decode_split(const void* q, int q_ld, const void* cache, const int* block_table,
                                    int max_blocks, const int* seq_lens, int S, int Hq, int Hkv, int D, int page,
                                    float scale, int window, void* out, int out_ld, int n_splits, void* workspace,
                                    long workspace_bytes, void* stream) {
  if (decode_checks(q, q_ld, cache, max_blocks, S, Hq, Hkv, D, page, window, out_ld)) return 1;
  int span = 0;
  if (split_checks(max_blocks, page, n_splits, &span)) return 1;
  DA_REQUIRE(workspace && (uintptr_t)workspace % 16 == 0 && workspace_bytes >= da_attn_decode_split_bytes(S, Hq, D, n_splits),
             "attn_decode_split: the workspace holds %ld bytes, %ld are needed", workspace_bytes,
             da_attn_decode_split_bytes(S, Hq, D, n_splits));
  if (S == 0) return 0;
  decode_launch(q, q_ld, cache, block_table, max_blocks, seq_lens, S, Hq, Hkv, D, page, scale, window, out, out_ld,
                n_splits, span, (float*)workspace, (hipStream_t)stream);
  DA_CHECK_LAUNCH("attn_decode_split");
  return 0;
}

// ---------------------------------------------------------------------------------------------
// The same without a workspace argument and without any allocation (see no_alloc.h).
// ---------------------------------------------------------------------------------------------
#include "no_alloc.h"
#include <mutex>

static __device__ __align__(256) unsigned char scratch[DA_DECODE_STATIC_SCRATCH_BYTES];

#define DA_MAX_DEVICES 64
static void* g_scratch_of_device[DA_MAX_DEVICES];      // the array's address on each GPU, asked for once
static std::mutex g_scratch_mutex;

// The address of `scratch` on the current device.  In host code the array's name is only a handle
// for the runtime; the memory's address differs from GPU to GPU and comes from hipGetSymbolAddress.
static int static_scratch(float** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  DA_REQUIRE(e == hipSuccess && dev >= 0 && dev < DA_MAX_DEVICES, "attn_decode_split_static: no current device (%s)",
             hipGetErrorString(e));
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_of_device[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    DA_REQUIRE(e == hipSuccess && p, "attn_decode_split_static: the scratch buffer's address is not known (%s)",
               hipGetErrorString(e));
    g_scratch_of_device[dev] = p;
  }
  *ptr = (float*)g_scratch_of_device[dev];
  return 0;
}

extern "C" int da_attn_decode_split_static(const void* q, int q_ld, const void* cache, const int* block_table,
                                           int max_blocks, const int* seq_lens, int S, int Hq, int Hkv, int D,
                                           int page, float scale, int window, void* out, int out_ld, int n_splits,
                                           void* stream) {
  if (decode_checks(q, q_ld, cache, max_blocks, S, Hq, Hkv, D, page, window, out_ld)) return 1;
  int span = 0;
  if (split_checks(max_blocks, page, n_splits, &span)) return 1;
  const long need = da_attn_decode_split_bytes(S, Hq, D, n_splits);
  DA_REQUIRE(need <= (long)DA_DECODE_STATIC_SCRATCH_BYTES,
             "attn_decode_split_static: %d sequences x %d heads x %d shares of head size %d need %ld bytes of scratch, "
             "the library holds %ld", S, Hq, n_splits, D, need, (long)DA_DECODE_STATIC_SCRATCH_BYTES);
  if (S == 0) return 0;
  float* partial = nullptr;
  if (static_scratch(&partial)) return 1;
  decode_launch(q, q_ld, cache, block_table, max_blocks, seq_lens, S, Hq, Hkv, D, page, scale, window, out, out_ld,
                n_splits, span, partial, (hipStream_t)stream);
  DA_CHECK_LAUNCH("attn_decode_split_static");
  return 0;
}

#endif  // DEC_REL
#endif
