// Paged attention in 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32): portions of prompts and one-token sequences alike.
//
// One workgroup per (sequence, query head, 16 query rows); 8 wavefronts share out the keys in aligned chunks of 32:
// wavefront v takes the chunks whose number is v modulo 8, in ascending order, with a running maximum and sum per row,
// and the wavefronts' partial results are merged in LDS in order.  Every sum's order so depends on a row's own position
// and the window only, never on how the step was cut or what else is in the batch; a chunk that a row does not see
// changes nothing in its sums.
//   scores : S[row, key] = Q . K^T, 2 pieces of 16 keys; a lane's 16-byte piece of a key row is 4 of the inner sum's
//            terms (an instruction takes the dimensions with d % 4 = j; see gemm_f32.hip for the fragments);
//   softmax: a lane holds 4 rows of one key column, so a row's maximum and sum are exchanges among 16 lanes;
//   values : stored dimension-major, so a lane's 16-byte piece is 4 consecutive keys of its dimension, which is the
//            right operand as it lies in memory; the weights turn from columns into rows through LDS.
// A compute unit takes four lanes' addresses at once where they lie in one line and one at a time else, and a fragment's neighbouring lanes
// are 16 different rows.  Head sizes above 64, whose values are asked for behind the scores, so load 64 consecutive bytes of a row by four
// neighbouring lanes (lane 4 c + q what lane c + 16 q multiplies), and a load's 64 pieces pass through 1 KB of LDS into their places, the
// same bits.  us, a row a lane / this, head size 128: 8 heads, 8 sequences of 1,000 keys in pages of 64 45.3 / 31.9, a prompt of 1,024
// 55.7 / 40.8; 12 heads, pages of 16, 4 prompts of 64 9.6 / 9.4, of 600 119 / 103, 16 sequences of 200 keys 11.9 / 11.3.  (Up to 64, where all loads are asked
// for at once, the way through LDS takes 0.3 us and gives it back only on a full chip: 4 sequences of 61 keys 5.4 / 5.7.)
// Up to a head size of 64 registers are held to 128, so that two workgroups share a compute unit; head size 64, us, one / two: 12 heads, 32 sequences of
// 30 keys 8.7 / 5.6, 64 of 600 43.7 / 39.3, two prompts of 1,024 73.7 / 58.5; 16 heads, prompts of 300 and 180 19.1 / 15.3, one of 600 24.5 / 21.1.  Not
// for prompts of up to 512 workgroups (ALONE: LDS that leaves no room for a second one), where two long ones meet on a compute unit while others have none: 8 heads, 600 14.7 / 16.2, 16 heads, 300
// 11.2 / 12.7, 12 heads, 300 and 180 13.1 / 14.4, 600 19.5 / 19.9.
// All key and value loads of a chunk are asked for before any is used (for head sizes up to 64; above, the values once
// the scores are done).  Bound by two trips to memory and D instructions of 32 cycles a chunk.  (Chunks of 64 keys leave most wavefronts
// of a short context without any and the others a chain twice as long; us, 64 / 32 keys a chunk, 12 heads of 64: 4 sequences of 61
// keys 7.4 / 5.7, of 200 9.2 / 8.0, 64 of 1,000 91 / 82, two prompts of 300 17.6 / 14.8, of 1,024 85 / 78; 8 heads, 8 of 1,000 keys 21.2 / 21.5; 6 heads of 32: a sequence of
// 61 keys 7.0 / 5.6, of 500 9.7 / 9.8, of 2,000 25.0 / 26.3.  One size for all contexts, so that a row's sums have one order.)
// Beside the plain kernel (attn_ref.hip), 8 heads, us at head size 64 / 128: a prompt of 1,024 589 -> 29 /
// 1,172 -> 50, 8 sequences of 1,000 keys 189 -> 21 / 379 -> 38.
// Formulas: core/src/main/java/io/teknek/deliverance/generator/CausalSelfAttention.java:481-491,512-527.
#include "gemm_common.h"
#include <da_read_arg.h>

#define AF_WAVES 8
#define AF_CHUNK 32
#define AF_PIECES (AF_CHUNK / 16)
#define AF_PLD (AF_CHUNK + 4)        // padded row of weights in LDS, floats

__device__ __forceinline__ floatx4 af_group(const float4& a, const float4& b, floatx4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}
__device__ __forceinline__ float af_max16(float v) {          // the maximum over 16 consecutive lanes, in all of them
  v = fmaxf(v, dpp_move<0xB1, 0xF>(v, v));
  v = fmaxf(v, dpp_move<0x4E, 0xF>(v, v));
  v = fmaxf(v, dpp_move<0x141, 0xF>(v, v));
  return fmaxf(v, dpp_move<0x140, 0xF>(v, v));
}

// Lane 4 c + q of N loads holds the piece of lane c + 16 q: through the wavefront's own part of LDS into their places, up to AF_TURN loads
// at a time.  (A row's pieces are turned by the row's group of four, so that the reads of 16 rows spread over the banks.  LDS serves a
// wavefront's instructions in order: it is the compiler alone that must keep them.)
#define AF_TURN 4
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
template <int N>
__device__ __forceinline__ void af_turn(float4 (&x)[N], f32x4_t* xs, int lane) {
  const int to = (lane & ~3) | ((lane & 3) ^ (lane / 16));
  const int from = 4 * (lane % 16) + ((lane / 16) ^ (lane % 16 / 4));
#pragma unroll
  for (int b = 0; b < N; b += AF_TURN) {
#pragma unroll
    for (int i = b; i < b + AF_TURN && i < N; ++i) xs[(i - b) * DA_WAVE + to] = __builtin_bit_cast(f32x4_t, x[i]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = b; i < b + AF_TURN && i < N; ++i) x[i] = __builtin_bit_cast(float4, xs[(i - b) * DA_WAVE + from]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// What the products cannot give: an entry whose weighted sum is not finite (the 16 rows of a tile share their keys, and a
// weight of zero times another row's infinite value is no number), or whose row has no weight at all (ll is 0: it sees no
// key, or only scores of minus infinity).  Key by key in ascending order, a value whose weight is zero is not looked at.
// Not on any ordinary row's way.  qr: the row's query; kb, vb: the head's keys and the entry's dimension in page 0; mm, ll:
// the row's maximum and sum.
__device__ __forceinline__ float af_entry(const float* qr, const float* kb, const float* vb, const int* bt, int lg, int pmask,
                                          long long page_elems, int D, int lo, int p, float scale, float mm, float ll) {
  if (ll != ll) return ll;
  bool any = false;
  float sum = 0.f;
  for (int key = lo; key <= p; ++key) {
    const int pg = bt[key >> lg];
    if (pg < 0) continue;
    any = true;
    if (ll == 0.f) break;
    const float* kr = kb + pg * page_elems + (key & pmask) * D;
    float dot = 0.f;
    for (int d = 0; d < D; ++d) dot = fmaf(qr[d], kr[d], dot);
    const float e = expf(dot * scale - mm);
    if (e != 0.f) sum = fmaf(e, vb[pg * page_elems + (key & pmask)], sum);
  }
  return ll == 0.f ? (any ? NAN : 0.f) : sum / ll;
}

template <int D16, bool ALONE = false>
__global__ void __launch_bounds__(AF_WAVES * DA_WAVE, D16 <= 4 ? 4 : 2)
attn_f32_kernel(const float* __restrict__ q, const float* __restrict__ cache, const int* __restrict__ block_table,
                const int* __restrict__ q_start, const int* __restrict__ seq_lens, int q_ld, int max_blocks, int Hq, int Hkv, int page,
                float scale, int window, float* __restrict__ out, int out_ld) {
  constexpr int D = D16 * 16;
  constexpr bool TURN = D16 > 4;
  constexpr int OLD = D + 4;                                   // padded row of a partial result
  constexpr int X_FLOATS = !TURN ? 0 : (D16 < AF_TURN ? D16 : AF_TURN) * DA_WAVE * 4, P_FLOATS = AF_WAVES * (16 * AF_PLD + X_FLOATS), O_FLOATS = AF_WAVES * 16 * OLD;
  constexpr int USED = P_FLOATS > O_FLOATS ? P_FLOATS : O_FLOATS, MORE_THAN_HALF = 81 * 1024 / 4;      // (of a compute unit's 160 KB)
  __shared__ __attribute__((aligned(16))) float smem[ALONE ? MORE_THAN_HALF : USED];   // weights and pieces on their way to their lanes, then partial results
  __shared__ float part_m[AF_WAVES][16], part_l[AF_WAVES][16];

  const int s = blockIdx.y, h = blockIdx.x, hk = Hq == Hkv ? h : h / (Hq / Hkv);
  const int t = threadIdx.x, lane = t % DA_WAVE, wave = __builtin_amdgcn_readfirstlane(t / DA_WAVE);
  const int col = lane % 16, quad = lane / 16;
  const int l_row = TURN ? lane / 4 : col, l_at = 4 * (TURN ? lane % 4 : quad);             // the row (of 16) and the first entry (of 16) that the lane loads
  const uint32_t k_at = 4u * (uint32_t)(l_row * D + l_at), v_at = 4u * (uint32_t)(l_row * page + l_at);      // bytes into a piece's keys and values
  const int* bt = block_table + (size_t)s * max_blocks;
  const int lg = 31 - __builtin_clz(page), pmask = page - 1;   // (a power of two, checked on the host)
  // Asked for side by side: the sequence's rows and length, and the pages of the chunk that this wavefront starts with where no window
  // cuts keys off (entries past the sequence's pages are read, the table has max_blocks of them, and never used).
  const int row0 = q_start[s], row1 = q_start[s + 1], len = seq_lens[s];
  int guess[AF_PIECES];
#pragma unroll
  for (int j = 0; j < AF_PIECES; ++j) {
    const int i = (wave * AF_CHUNK + j * 16) >> lg;
    guess[j] = bt[i < max_blocks ? i : max_blocks - 1];
  }
  da_read_arg(scale);
  da_read_arg(out);
  da_read_arg(out_ld);
  const int T = row1 - row0;
  const int i0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * 16;  // (the rows with the most keys are launched first)
  if (i0 >= T) return;
  const int past = len - T;
  const int last_row = i0 + 15 < T ? i0 + 15 : T - 1;
  const int p_max = past + last_row;                           // the last key that any of the rows sees (-1: a padding row)
  const int lo_min = (window > 0 && past + i0 - window + 1 > 0) ? past + i0 - window + 1 : 0;
  const long long page_elems = 2LL * Hkv * page * D;
  const float* kbase = cache + (long long)hk * page * D;
  const float* vbase = cache + (long long)(Hkv + hk) * page * D;

  float4 qf[D16];
  bool q_placed = !TURN || last_row == i0;                              // (one row: the same piece for all lanes of a quarter, read as it is used)
  {
    const int qi = i0 + l_row < T ? i0 + l_row : T - 1;
    const float* qr = q + (size_t)(row0 + qi) * q_ld + h * D + (q_placed ? quad * 4 : l_at);
#pragma unroll
    for (int g = 0; g < D16; ++g) qf[g] = *(const float4*)(qr + g * 16);
  }
  floatx4 o[D16];
#pragma unroll
  for (int d = 0; d < D16; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m[4], l[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) { m[r] = -INFINITY; l[r] = 0.f; }
  float* const ps = smem + wave * 16 * AF_PLD;
  f32x4_t* const xs = (f32x4_t*)(smem + AF_WAVES * 16 * AF_PLD + wave * X_FLOATS);

  const int first_chunk = lo_min / AF_CHUNK;
  for (int ci = first_chunk + (wave + AF_WAVES - first_chunk % AF_WAVES) % AF_WAVES; ci * AF_CHUNK <= p_max; ci += AF_WAVES) {
    const int c0 = ci * AF_CHUNK;
    // The pages of the chunk's pieces of 16 keys (a piece lies in one page), the same for the whole wavefront.  A piece
    // that no row sees, or whose page was given back, reads page 0 and is dropped.
    bool seen[AF_PIECES];
    const float* kp[AF_PIECES];
    const float* vp[AF_PIECES];
#pragma unroll
    for (int j = 0; j < AF_PIECES; ++j) {
      const int k0 = c0 + j * 16;
      const bool in = k0 <= p_max && k0 + 15 >= lo_min;
      const int pg = !in ? -1 : (ci == wave ? __builtin_amdgcn_readfirstlane(guess[j]) : __builtin_amdgcn_readfirstlane(bt[k0 >> lg]));
      seen[j] = pg >= 0;
      const long long off = (long long)(pg >= 0 ? pg : 0) * page_elems;
      kp[j] = kbase + off + (k0 & pmask) * D;
      vp[j] = vbase + off + (k0 & pmask);
    }
    float4 kf[AF_PIECES][D16], vf[AF_PIECES][D16];
    constexpr bool EARLY_V = D16 <= 4;
#pragma unroll
    for (int j = 0; j < AF_PIECES; ++j)
#pragma unroll
      for (int g = 0; g < D16; ++g) kf[j][g] = *(const float4*)((const char*)(kp[j] + g * 16) + k_at);
    if (EARLY_V) {
#pragma unroll
      for (int j = 0; j < AF_PIECES; ++j)
#pragma unroll
        for (int d = 0; d < D16; ++d) vf[j][d] = *(const float4*)((const char*)(vp[j] + d * 16 * page) + v_at);
    }
    __builtin_amdgcn_sched_barrier(0);                          // (the loads stay ahead of the arithmetic)
    if (TURN && !q_placed) {                                            // (not in front of the loop, where the keys would be asked for behind it)
      af_turn(qf, xs, lane);
      q_placed = true;
    }
    floatx4 sc[AF_PIECES];
#pragma unroll
    for (int j = 0; j < AF_PIECES; ++j) {
      if (TURN) af_turn(kf[j], xs, lane);
      sc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < D16; ++g) sc[j] = af_group(qf[g], kf[j][g], sc[j]);
    }
    float alpha[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + quad * 4 + r, p = past + i;
      const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
      bool ok[AF_PIECES];
      float top = -INFINITY;
#pragma unroll
      for (int j = 0; j < AF_PIECES; ++j) {
        const int key = c0 + j * 16 + col;
        ok[j] = seen[j] && i < T && key <= p && key >= lo;
        sc[j][r] = ok[j] ? sc[j][r] * scale : -INFINITY;        // (a select: an unseen key's row may hold anything)
        top = fmaxf(top, sc[j][r]);
      }
      const float m_new = fmaxf(m[r], af_max16(top));
      alpha[r] = m_new == -INFINITY ? 1.f : expf(m[r] - m_new);
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;     // (scores of minus infinity alone weigh nothing here: another chunk may hold more)
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < AF_PIECES; ++j) {
        const float e = ok[j] ? expf(sc[j][r] - m_ref) : 0.f;
        ps[(quad * 4 + r) * AF_PLD + j * 16 + col] = e;
        sum += e;
      }
      l[r] = l[r] * alpha[r] + group_sum<16>(sum);
      m[r] = m_new;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
    for (int d = 0; d < D16; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[d][r] *= alpha[r];
    if (!EARLY_V) {
#pragma unroll
      for (int j = 0; j < AF_PIECES; ++j)
#pragma unroll
        for (int d = 0; d < D16; ++d) vf[j][d] = *(const float4*)((const char*)(vp[j] + d * 16 * page) + v_at);
    }
#pragma unroll
    for (int j = 0; j < AF_PIECES; ++j) {
      const float4 w = *(const float4*)&ps[col * AF_PLD + j * 16 + quad * 4];
      if (TURN) af_turn(vf[j], xs, lane);
      // keys past the last seen one were never written and keys in front of a window may be anybody's: zeros in their
      // place (their weights are zero, but zero times an infinity is not)
      const int k0 = c0 + j * 16 + quad * 4;
#pragma unroll
      for (int d = 0; d < D16; ++d) {
        float4 v = vf[j][d];
        v.x = seen[j] && k0 <= p_max && k0 >= lo_min ? v.x : 0.f;
        v.y = seen[j] && k0 + 1 <= p_max && k0 + 1 >= lo_min ? v.y : 0.f;
        v.z = seen[j] && k0 + 2 <= p_max && k0 + 2 >= lo_min ? v.z : 0.f;
        v.w = seen[j] && k0 + 3 <= p_max && k0 + 3 >= lo_min ? v.w : 0.f;
        o[d] = af_group(w, v, o[d]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
  __syncthreads();                                              // the weights' place takes the partial results
#pragma unroll
  for (int d = 0; d < D16; ++d)
#pragma unroll
    for (int r = 0; r < 4; ++r) smem[(wave * 16 + quad * 4 + r) * OLD + d * 16 + col] = o[d][r];
  if (col == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) { part_m[wave][quad * 4 + r] = m[r]; part_l[wave][quad * 4 + r] = l[r]; }
  }
  __syncthreads();
  for (int e = t; e < 16 * D; e += AF_WAVES * DA_WAVE) {
    const int row = e / D, d = e % D;
    if (i0 + row >= T) continue;
    float mm = part_m[0][row];
#pragma unroll
    for (int w = 1; w < AF_WAVES; ++w) mm = fmaxf(mm, part_m[w][row]);
    float ll = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
      const float f = part_m[w][row] == -INFINITY ? 0.f : expf(part_m[w][row] - mm);
      ll += part_l[w][row] * f;
      v += smem[(w * 16 + row) * OLD + d] * f;
    }
    float* const entry = out + (size_t)(row0 + i0 + row) * out_ld + h * D + d;
    if (ll > 0.f && fabsf(v) < INFINITY) {
      *entry = v / ll;
      continue;
    }
    const int p = past + i0 + row;
    *entry = af_entry(q + (size_t)(row0 + i0 + row) * q_ld + h * D, kbase, vbase + (long long)d * page, bt, lg, pmask, page_elems, D,
                      (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0, p, scale, mm, ll);
  }
}

// Attention of every row of a step (sequence s has the rows q_start[s] .. q_start[s + 1] - 1, the last of which sits at
// position seq_lens[s] - 1; at most max_query_len rows) over its sequence's pages.
extern "C" int da_attn_f32(const float* q, int q_ld, const float* cache, const int* block_table, int max_blocks, const int* q_start,
                           const int* seq_lens, int n_seqs, int max_query_len, int Hq, int Hkv, int D, int page, float scale, int window,
                           float* out, int out_ld, void* stream) {
  DA_REQUIRE(n_seqs >= 0 && max_query_len > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0, "attn_f32: bad sizes (%d sequences, %d rows, %d and %d heads)",
             n_seqs, max_query_len, Hq, Hkv);
  DA_REQUIRE(D % 16 == 0 && D >= 16 && D <= 128, "attn_f32: head size %d is not a multiple of 16 up to 128", D);
  DA_REQUIRE(page % 16 == 0 && (page & (page - 1)) == 0, "attn_f32: page size %d must be a power of two from 16 on", page);
  DA_REQUIRE(q_ld >= Hq * D && out_ld >= Hq * D && q_ld % 4 == 0, "attn_f32: row lengths (q %d, out %d)", q_ld, out_ld);
  DA_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)cache % 16 == 0, "attn_f32: q and the cache must be 16-byte aligned");
  DA_REQUIRE(window >= 0 && max_blocks > 0, "attn_f32: bad window or block table");
  if (n_seqs == 0) return 0;
  // (a head and a sequence a workgroup, found without a division; a launch's second size ends at 65,535)
  for (int s0 = 0; s0 < n_seqs; s0 += 65535) {
    const int n = n_seqs - s0 < 65535 ? n_seqs - s0 : 65535;
    const long workgroups = (long)Hq * n * da_ceil_div(max_query_len, 16);
    const bool two = workgroups > 512 || (max_query_len <= 16 && workgroups > 256);
    const dim3 grid(Hq, n, da_ceil_div(max_query_len, 16)), block(AF_WAVES * DA_WAVE);
#define AF_LAUNCH(...)                                                                                                                     \
  hipLaunchKernelGGL((attn_f32_kernel<__VA_ARGS__>), grid, block, 0, (hipStream_t)stream, q, cache, block_table + (size_t)s0 * max_blocks, q_start + s0, \
                     seq_lens + s0, q_ld, max_blocks, Hq, Hkv, page, scale, window, out, out_ld)
    switch (D / 16) {
      case 1: AF_LAUNCH(1); break;
      case 2: AF_LAUNCH(2); break;
      case 3: AF_LAUNCH(3); break;
      case 4: if (two) AF_LAUNCH(4); else AF_LAUNCH(4, true); break;
      case 5: AF_LAUNCH(5); break;
      case 6: AF_LAUNCH(6); break;
      case 7: AF_LAUNCH(7); break;
      default: AF_LAUNCH(8); break;
    }
#undef AF_LAUNCH
  }
  DA_CHECK_LAUNCH("attn_f32");
  return 0;
}
