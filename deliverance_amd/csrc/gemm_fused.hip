// Decode-sized fused product: LayerNorm of the 32-bit residual rows, the bfloat16 product on the
// matrix cores, bias / activation, and (for a q|k|v projection) the write of the new keys and
// values into the paged cache -- one kernel where a step with a handful of rows would otherwise
// pay for three.
//
//   a[m, :]   = LayerNorm(x[rows ? rows[m] : m, :]) rounded to bf16      (32-bit statistics)
//   out[m, n] = act( sum_k a[m, k] * w[n, k] + bias[n] )
//   columns n >= kv.q_cols of a q|k|v projection are also stored to the cache row kv.slot_map[m]
//
// Every workgroup owns a few output columns and all rows, and computes the statistics of
// all rows itself (M * K floats from L2: cheap while M is small; the host uses the unfused
// kernels for larger steps): mean, then the centred sum of squares.  Three kernels: gemm_ln_quads (a wavefront
// holds a part of every row, the parts' statistics are joined), gemm_ln_rows (a wavefront a row or two, held in registers) and
// gemm_ln_skinny (any of up to 32 rows, parameters of unlike dtypes).
// Formulas: core/src/main/java/io/teknek/deliverance/generator/LayerNorm.java:127-150,
// CausalSelfAttention.java:266-291,315-336, MLPBlock.java:250-292.
#include "gemm_common.h"
#include <da_read_arg.h>
#include <da_lane_swap.h>

#define FZ_COLS 16
#define FZ_VPL 8          // float4 per lane when a row is held in registers: K <= 2048

struct LnPrologue {
  const float* x;
  const int* rows;
  const void* g;
  int g_dtype;
  const void* b;
  int b_dtype;
  float eps;
  // LayerNorm: center 1, gain_offset 0.  A root-mean-square norm is the same arithmetic with the mean taken
  // as zero (center 0), no bias, and a gain of gain_offset + g (1 + g for gains stored around zero).
  float center;
  float gain_offset;
};

__device__ __forceinline__ void load8_param(const void* p, int dtype, int i, float* o) {
  if (dtype == DA_BF16) {
    const uint4 u = *(const uint4*)((const bf16_t*)p + i);
    const uint32_t v[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[2 * e] = __uint_as_float(v[e] << 16);
      o[2 * e + 1] = __uint_as_float(v[e] & 0xffff0000u);
    }
  } else {
    const float4 a = *(const float4*)((const float*)p + i), c = *(const float4*)((const float*)p + i + 4);
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = c.x; o[5] = c.y; o[6] = c.z; o[7] = c.w;
  }
}

template <int MT, int NW, int FZ_UNROLL>
// (for one row tile the registers are held to 128, so that two workgroups of 8 wavefronts share a compute unit)
__global__ void __launch_bounds__(NW * 64, MT == 1 ? 4 : 1)
gemm_ln_skinny_kernel(LnPrologue ln, const bf16_t* __restrict__ w, int ldw, Epilogue ep, KvScatter kv,
                      int M, int N, int K) {
  __shared__ float red[NW][MT * 16][FZ_COLS + 1];
  __shared__ float s_mean[MT * 16], s_rstd[MT * 16];
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int n0 = blockIdx.x * FZ_COLS;
  const int fr = lane % 16, fk = (lane / 16) * 8;

  // The first chunks of w and of the norm's gain and bias do not depend on the statistics: their
  // loads are issued first and fly while the rows are read and reduced.
  const uint4 zero = make_uint4(0, 0, 0, 0);
  const bool wrow_ok = n0 + fr < N;
  const bf16_t* wp = w + (size_t)(wrow_ok ? n0 + fr : 0) * ldw + fk;
  uint4 wv[FZ_UNROLL];
  float gg[FZ_UNROLL][8], bb[FZ_UNROLL][8];
  auto load_wgb = [&](int k0) {
#pragma unroll
    for (int u = 0; u < FZ_UNROLL; ++u) {
      const int k = k0 + u * NW * 32;
      const bool kin = k + fk < K;
      const int ks = kin ? k : -fk;
      wv[u] = load16(wp + ks);      // past K: the row's first chunk, met by zeros in a; past N: row 0, never stored
      load8_param(ln.g, ln.g_dtype, ks + fk, gg[u]);
      if (ln.b) load8_param(ln.b, ln.b_dtype, ks + fk, bb[u]);
    }
  };
  load_wgb(wave * 32);
  // what the epilogue needs, also early: this thread's output elements are e = t, t + THREADS, ...
  constexpr int EPT = (MT * 16 * FZ_COLS + NW * 64 - 1) / (NW * 64);
  float e_bias[EPT];
  int e_slot[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = t + j * NW * 64, em = e / FZ_COLS, ec = e % FZ_COLS;
    const bool ok = e < MT * 16 * FZ_COLS && em < M && n0 + ec < N;
    e_bias[j] = (ok && ep.bias) ? load_param(ep.bias, ep.bias_dtype, n0 + ec) : 0.f;
    e_slot[j] = (ok && kv.cache) ? kv.slot_map[em] : -1;
  }

  // ---- statistics of every row: wavefront v takes rows v, v + NW, ...
  for (int m = wave; m < M; m += NW) {
    const float* xr = ln.x + (size_t)(ln.rows ? ln.rows[m] : m) * K;
    float4 v[FZ_VPL];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < FZ_VPL; ++i) {
      const int c = (lane + i * 64) * 4;
      v[i] = *(const float4*)(xr + (c < K ? c : 0));          // never a conditional load, nor a value replaced
      s += (c < K ? 1.f : 0.f) * ((v[i].x + v[i].y) + (v[i].z + v[i].w));
    }
    const float mean = wave_sum(s) / (float)K * ln.center;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < FZ_VPL; ++i) {
      const int c = (lane + i * 64) * 4;
      if (c < K) {
        const float d0 = v[i].x - mean, d1 = v[i].y - mean, d2 = v[i].z - mean, d3 = v[i].w - mean;
        q += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
      }
    }
    const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)K + ln.eps);
    if (lane == 0) { s_mean[m] = mean; s_rstd[m] = rstd; }
  }
  lds_barrier();

  floatx4 acc[MT];
  float mean[MT], rstd[MT];
  bool arow_ok[MT];
  const float* xp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int m = i * 16 + fr;
    arow_ok[i] = m < M;
    const int ms = arow_ok[i] ? m : 0;
    mean[i] = s_mean[ms]; rstd[i] = s_rstd[ms];
    xp[i] = ln.x + (size_t)(ln.rows ? ln.rows[ms] : ms) * K + fk;
  }

  for (int k0 = wave * 32; k0 < K; k0 += NW * 32 * FZ_UNROLL) {
    if (k0 != wave * 32) load_wgb(k0);
    float4 xa[FZ_UNROLL][MT][2];
#pragma unroll
    for (int u = 0; u < FZ_UNROLL; ++u) {
      const int k = k0 + u * NW * 32;
      const int ks = (k + fk < K) ? k : -fk;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        xa[u][i][0] = *(const float4*)(xp[i] + ks);
        xa[u][i][1] = *(const float4*)(xp[i] + ks + 4);
      }
    }
#pragma unroll
    for (int u = 0; u < FZ_UNROLL; ++u) {
      const int k = k0 + u * NW * 32;
      const bool kin = k + fk < K;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float xs[8] = {xa[u][i][0].x, xa[u][i][0].y, xa[u][i][0].z, xa[u][i][0].w,
                             xa[u][i][1].x, xa[u][i][1].y, xa[u][i][1].z, xa[u][i][1].w};
        uint32_t pk[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float y0 = (xs[2 * e] - mean[i]) * rstd[i] * (gg[u][2 * e] + ln.gain_offset);
          float y1 = (xs[2 * e + 1] - mean[i]) * rstd[i] * (gg[u][2 * e + 1] + ln.gain_offset);
          if (ln.b) { y0 += bb[u][2 * e]; y1 += bb[u][2 * e + 1]; }
          pk[e] = (uint32_t)f32_to_bf16(y0) | ((uint32_t)f32_to_bf16(y1) << 16);
        }
        uint4 av = make_uint4(pk[0], pk[1], pk[2], pk[3]);
        if (!(kin && arow_ok[i])) av = zero;
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av),
                                                         __builtin_bit_cast(bf16x8_t, wv[u]), acc[i], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][i * 16 + 4 * (lane / 16) + r][fr] = acc[i][r];
  lds_barrier();
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = t + j * NW * 64, em = e / FZ_COLS, ec = e % FZ_COLS, n = n0 + ec;
    if (!(e < MT * 16 * FZ_COLS && em < M && n < N)) continue;
    float v = red[0][em][ec];
#pragma unroll
    for (int v2 = 1; v2 < NW; ++v2) v += red[v2][em][ec];
    epilogue_store(ep, em, n, v, e_bias[j]);
    if (kv.cache) kv_column_store(kv, kv_column(kv, n), e_slot[j], apply_act_bf16(v + e_bias[j], ep.act));
  }
}

struct LnRest {
  float eps, center, gain_offset;
};

// ---------------------------------------------------------------------------------------------
// M <= 8, K <= 2048, parameters of one dtype.  MFMA 16x16x32 with pieces of k side by side (gemm_skinny4 in gemm_mfma.hip): a lane holds 8
// consecutive k of row r4 of 4 of w and of 4 rows of x, four neighbouring lanes 64 consecutive bytes, and what it holds of x is what it
// normalises: nothing passes through LDS but a wavefront's mean and squares of each row.  Wavefront v of NW has the steps v and, SW of them, v + NW of 128
// elements of k.  A row's statistics join its wavefronts' means and squares around them (M2 = sum of M2_v + n_v (mean_v - mean)^2).
// Bound by what a wavefront computes for each row (so as few wavefronts as hold k in two steps each: K = 768, 3,072 columns, one row 3.5 us with 6
// of them, 2.9 with 3) and by the bytes of w.  A workgroup owns `cols` columns, 4 * NG at most.  Beside gemm_ln_rows below: ln_quads_takes.
// (w alone, read and dropped: 2.5 at K = 768, 4.5 to 5 and 5.2 at 1,600.)
// ---------------------------------------------------------------------------------------------
template <int MG, int NG, int NW, int SW, bool PBF16>
__global__ void __launch_bounds__(NW * 64)
gemm_ln_quads_kernel(const float* __restrict__ x, const int* __restrict__ rows, const void* __restrict__ gain, const void* __restrict__ shift,
                     const bf16_t* __restrict__ w, int ldw, int N, int K, int rows_cols, LnRest lr_, Epilogue ep, KvScatter kv) {
  const int M = rows_cols & 0xff, cols = rows_cols >> 8;
  constexpr int ROWS = 4 * MG, COLS = 4 * NG;
  __shared__ float2 stats[NW][ROWS];
  __shared__ float red[NW][ROWS][COLS + 1];
  const int t = threadIdx.x, lane = t % 64, wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int n0 = blockIdx.x * cols;
  const int n_end = n0 + cols < N ? n0 + cols : N;
  const int r4 = lane / 4 % 4, kb = (4 * (lane / 16) + lane % 4) * 8;
  // ---- all loads first, in the order of their use (lanes past K read their rows' first piece, lanes past M or the last column the first row)
  constexpr int PH = PBF16 ? 1 : 2;                  // 16-byte pieces of a lane's 8 gains
  float4 xv[SW][MG][2];
  uint4 gq[SW][PH], bq[SW][PH], wv[SW][NG];
  const float* xr[MG];
#pragma unroll
  for (int i = 0; i < MG; ++i) {
    const int m = 4 * i + r4 < M ? 4 * i + r4 : 0;
    xr[i] = x + (size_t)(rows ? rows[m] : m) * K;
  }
#pragma unroll
  for (int u = 0; u < SW; ++u) {
    const int k = (wave + u * NW) * 128 + kb, ks = k < K ? k : 0;
#pragma unroll
    for (int i = 0; i < MG; ++i) {
      xv[u][i][0] = *(const float4*)(xr[i] + ks);
      xv[u][i][1] = *(const float4*)(xr[i] + ks + 4);
    }
  }
#pragma unroll
  for (int u = 0; u < SW; ++u) {
    const int k = (wave + u * NW) * 128 + kb, ks = k < K ? k : 0;
    const void* sh = shift ? shift : gain;
#pragma unroll
    for (int h = 0; h < PH; ++h) {
      gq[u][h] = *(const uint4*)((const char*)gain + (size_t)(ks + 4 * h) * (PBF16 ? 2 : 4));
      bq[u][h] = *(const uint4*)((const char*)sh + (size_t)(ks + 4 * h) * (PBF16 ? 2 : 4));
    }
  }
#pragma unroll
  for (int u = 0; u < SW; ++u) {
    const int k = (wave + u * NW) * 128 + kb, ks = k < K ? k : 0;
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int n = n0 + 4 * j + r4;
      wv[u][j] = load16(w + (size_t)(n < n_end ? n : n0) * ldw + ks);
    }
  }
  // this thread's output element, with what its epilogue needs
  static_assert(ROWS * COLS <= NW * 64, "an output element a thread");
  const int em = t / COLS, ec = t % COLS, en = n0 + ec;
  const bool e_ok = em < M && en < n_end;                             // (M is ROWS at most)
  const void* e_bsrc = ep.bias ? ep.bias : (const void*)w;
  const int e_slot = kv.cache ? kv.slot_map[e_ok ? em : 0] : -1;
  const int e_bidx = (ep.bias && e_ok) ? en : 0;
  const uint32_t e_bias_raw = PBF16 ? (uint32_t)((const bf16_t*)e_bsrc)[e_bidx] : ((const uint32_t*)e_bsrc)[e_bidx];
  da_read_arg(ep.act);
  da_read_arg(ep.out_dtype);
  KvColumn e_col;
  if (kv.cache) e_col = kv_column(kv, en);
  __builtin_amdgcn_sched_barrier(0);

  // ---- statistics: a wavefront's own mean and squares around it, joined in the order of the wavefronts
  auto count = [&](int v) {                            // elements of a row that wavefront v holds
    int n = K - v * 128;
    n = n < 0 ? 0 : (n < 128 ? n : 128);
#pragma unroll
    for (int u = 1; u < SW; ++u) {
      int n2 = K - (v + u * NW) * 128;
      n += n2 < 0 ? 0 : (n2 < 128 ? n2 : 128);
    }
    return n;
  };
  const int mine = count(wave);
  const float inv_mine = mine > 0 ? lr_.center / (float)mine : 0.f;
#pragma unroll
  for (int i = 0; i < MG; ++i) {
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < SW; ++u) {
      const float in = (wave + u * NW) * 128 + kb < K ? 1.f : 0.f;
      const float4 p = xv[u][i][0], q = xv[u][i][1];
      s += in * (((p.x + p.y) + (p.z + p.w)) + ((q.x + q.y) + (q.z + q.w)));
    }
    const float mean = quarter_sum(group_sum<4>(s)) * inv_mine;
    float m2 = 0.f;
#pragma unroll
    for (int u = 0; u < SW; ++u) {
      const float in = (wave + u * NW) * 128 + kb < K ? 1.f : 0.f;
      const float4 p = xv[u][i][0], q = xv[u][i][1];
      const float d[8] = {p.x - mean, p.y - mean, p.z - mean, p.w - mean, q.x - mean, q.y - mean, q.z - mean, q.w - mean};
      m2 += in * (((d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3])) + ((d[4] * d[4] + d[5] * d[5]) + (d[6] * d[6] + d[7] * d[7])));
    }
    m2 = quarter_sum(group_sum<4>(m2));
    if (lane < 16 && lane % 4 == 0) stats[wave][4 * i + r4] = make_float2(mean, m2);
  }
  lds_barrier();
  // ---- the normalised rows, straight into fragments, and the products
  floatx4 acc[MG][NG];
  const float inv_k = 1.0f / (float)K;
#pragma unroll
  for (int i = 0; i < MG; ++i) {
    float2 st[NW];
#pragma unroll
    for (int v = 0; v < NW; ++v) st[v] = stats[v][4 * i + r4];
    float mean = 0.f;
#pragma unroll
    for (int v = 0; v < NW; ++v) mean += (float)count(v) * st[v].x;
    mean *= inv_k;
    float m2 = 0.f;
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      const float d = st[v].x - mean;
      m2 += st[v].y + (float)count(v) * d * d;
    }
    const float rstd = 1.0f / sqrtf(m2 * inv_k + lr_.eps);
#pragma unroll
    for (int j = 0; j < NG; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < SW; ++u) {
      const bool in = (wave + u * NW) * 128 + kb < K;
      const float4 p = xv[u][i][0], q = xv[u][i][1];
      const float xs[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
      float g8[8], b8[8];
      if (PBF16) {
        const uint32_t gw[4] = {gq[u][0].x, gq[u][0].y, gq[u][0].z, gq[u][0].w}, bw[4] = {bq[u][0].x, bq[u][0].y, bq[u][0].z, bq[u][0].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          g8[2 * e] = __uint_as_float(gw[e] << 16); g8[2 * e + 1] = __uint_as_float(gw[e] & 0xffff0000u);
          b8[2 * e] = __uint_as_float(bw[e] << 16); b8[2 * e + 1] = __uint_as_float(bw[e] & 0xffff0000u);
        }
      } else {
        const uint4 g0 = gq[u][0], g1 = gq[u][PH - 1], b0 = bq[u][0], b1 = bq[u][PH - 1];
        const uint32_t gw[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w}, bw[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) { g8[e] = __uint_as_float(gw[e]); b8[e] = __uint_as_float(bw[e]); }
      }
      uint32_t pk[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float y0 = (xs[2 * e] - mean) * rstd * (g8[2 * e] + lr_.gain_offset), y1 = (xs[2 * e + 1] - mean) * rstd * (g8[2 * e + 1] + lr_.gain_offset);
        if (shift) { y0 += b8[2 * e]; y1 += b8[2 * e + 1]; }
        pk[e] = in ? pack2_bf16(y0, y1) : 0u;
      }
      const uint4 av = make_uint4(pk[0], pk[1], pk[2], pk[3]);
#pragma unroll
      for (int j = 0; j < NG; ++j) {
        const uint4 wz = in ? wv[u][j] : make_uint4(0, 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wz), __builtin_bit_cast(bf16x8_t, av), acc[i][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MG; ++i)
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const float d01 = lane & 1 ? acc[i][j][1] : acc[i][j][0], d23 = lane & 1 ? acc[i][j][3] : acc[i][j][2];
      const float v = group_sum<4>(lane & 2 ? d23 : d01);
      if (lane % 4 == 0) red[wave][4 * i + r4][j * 4 + lane / 16] = v;
    }
  lds_barrier();
  if (e_ok) {
    float v = red[0][em][ec];
#pragma unroll
    for (int v2 = 1; v2 < NW; ++v2) v += red[v2][em][ec];
    const float e_bias = !ep.bias ? 0.f : (PBF16 ? __uint_as_float(e_bias_raw << 16) : __uint_as_float(e_bias_raw));
    epilogue_store(ep, em, en, v, e_bias);
    if (kv.cache) kv_column_store(kv, e_col, e_slot, apply_act_bf16(v + e_bias, ep.act));
  }
}

// ---------------------------------------------------------------------------------------------
// Up to 8 rows and K = 1,536, up to 16 and 1,024 (what ln_quads_takes leaves of them), parameters of one dtype: every load in whole cache lines.
// Wavefront v of 8 reads rows v and v + 8 whole (RV float4 a lane), with the gain and bias at the
// same places, computes their statistics, and writes the normalised rows as bfloat16 into LDS,
// zeros past K.  The steps of w (64 elements of k, 8 rows x 128 bytes a load; wavefront v takes the
// steps v, v + 8, ...) are asked for before anything else is computed and parked in the wavefront's
// own piece of LDS; the fragments of both operands are read from LDS.  Steps past K read step 0 and
// meet zeros.  The sum over k runs in the order of the steps, whatever M is.
// TWO_ROWS false: M <= 8, a wavefront has one row and LDS holds 8 (the fragment's rows 8..15 read
// rows 0..7 again and are never stored): half the LDS, so that with a wide K two workgroups still
// share a compute unit and N / 16 workgroups run side by side.
// ---------------------------------------------------------------------------------------------
#define FL_LD (64 + 8)       // padded row of a parked step of w, elements
// A workgroup owns `cols` columns, 16 * CT at most.  16 of them leave some compute units with more workgroups than others
// where there are more than 256: the launch then takes as many columns (CT 2) as give every compute unit one workgroup, or
// two.  A compute unit pulls in about 70 GB/s at best, so its bytes are
// what the kernel takes: rows of w, the rows of x, and gain and bias once a wavefront that has a row.
// The arguments that the loads need are the first 14 words (build.py: KERNARG_PRELOAD; M and cols, 16 and 32 at most, share one);
// what the epilogue needs is asked for behind the operands, with the place in the cache of the thread's column.
template <int RV, bool PBF16, bool TWO_ROWS, int CT>
__global__ void __launch_bounds__(512)
gemm_ln_rows_kernel(const float* __restrict__ x, const int* __restrict__ rows, const void* __restrict__ gain, const void* __restrict__ shift,
                    const bf16_t* __restrict__ w, int ldw, int N, int K, int rows_cols, LnRest lr_, Epilogue ep, KvScatter kv) {
  const int M = rows_cols & 0xff, cols = rows_cols >> 8;
  const LnPrologue ln{x, rows, gain, 0, shift, 0, lr_.eps, lr_.center, lr_.gain_offset};
  constexpr int NW = 8, KMAX = RV * 256, ALD = KMAX + 8;      // ALD: padded row of a in LDS, elements
  constexpr int SW = (RV * 4 + NW - 1) / NW;                   // steps a wavefront
  constexpr int RPW = TWO_ROWS ? 2 : 1, AR = RPW * NW;         // rows a wavefront normalises; rows in LDS
  __shared__ __attribute__((aligned(16))) bf16_t a_lds[AR][ALD];
  constexpr int COLS = CT * 16, WL = COLS / 8;                 // columns at most; loads of 8 rows that cover w's
  // The wavefronts' sums lie behind the parked steps, where two workgroups still share a compute unit; else they take their place once all
  // products are done, behind a barrier more.
  constexpr int STAGE_BYTES = NW * COLS * FL_LD * 2, RED_BYTES = NW * 16 * (COLS + 1) * 4;
  constexpr bool APART = AR * ALD * 2 + STAGE_BYTES + RED_BYTES <= 80 * 1024;
  __shared__ __attribute__((aligned(16))) char stage_red[APART ? STAGE_BYTES + RED_BYTES : (STAGE_BYTES > RED_BYTES ? STAGE_BYTES : RED_BYTES)];
  bf16_t (*stage)[COLS * FL_LD] = (bf16_t (*)[COLS * FL_LD])stage_red;
  float (*red)[16][COLS + 1] = (float (*)[16][COLS + 1])(stage_red + (APART ? STAGE_BYTES : 0));
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int n0 = blockIdx.x * cols;                  // the workgroup's columns: n0 .. n_end - 1
  const int n_end = n0 + cols < N ? n0 + cols : N;
  const int fr = lane % 16, fk = (lane / 16) * 8;    // a fragment: row fr of 16, k-group lane / 16
  const int lr = lane / 8, lc = (lane % 8) * 8;      // a load of w: row lr of 8, 16-byte piece lane % 8

  // ---- all loads first, in the order of their use
  // (rows from M on are neither read nor normalised: what they give is never stored; the row number
  // is made a scalar so that the branch around their loads is one for the whole wavefront)
  const int row0 = __builtin_amdgcn_readfirstlane(wave);
  float4 sv[RPW][RV];
  uint4 gq[RV], bq[RV];                              // gain and bias at this lane's places (bfloat16: .x .y only)
  auto load_row = [&](float4 (&v)[RV], int m) {
    const float* xr = ln.x + (size_t)(ln.rows ? ln.rows[m] : m) * K;
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const int c = (lane + i * 64) * 4;
      v[i] = *(const float4*)(xr + (c < K ? c : 0));
    }
  };
  if (row0 < M) {                                    // (a wavefront without a row needs no gain and bias either)
    load_row(sv[0], row0);
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const int c = (lane + i * 64) * 4, cs = c < K ? c : 0;
      if (PBF16) {
        const uint2 g2 = *(const uint2*)((const bf16_t*)ln.g + cs);
        gq[i] = make_uint4(g2.x, g2.y, 0, 0);
        const uint2 b2 = *(const uint2*)((const bf16_t*)(ln.b ? ln.b : ln.g) + cs);
        bq[i] = make_uint4(b2.x, b2.y, 0, 0);
      } else {
        gq[i] = *(const uint4*)((const float*)ln.g + cs);
        bq[i] = *(const uint4*)((const float*)(ln.b ? ln.b : ln.g) + cs);
      }
    }
    if (TWO_ROWS && row0 + NW < M) load_row(sv[RPW - 1], row0 + NW);
  }
  uint4 wv[SW][WL];
#pragma unroll
  for (int u = 0; u < SW; ++u) {
    const int k0 = (wave + u * NW) * 64;
    const int kk = k0 + lc < K ? k0 + lc : 0;        // past K: the row's first piece
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int n = n0 + i * 8 + lr;
      wv[u][i] = load16(w + (size_t)(n < n_end ? n : n0) * ldw + kk);
    }
  }
  // this thread's output element (16 x COLS of them, a thread one at most), with what its epilogue needs
  static_assert(16 * COLS <= NW * 64, "an output element a thread");
  const int em = t / COLS, ec = t % COLS, en = n0 + ec;
  const bool e_ok = em < 16 && em < M && en < n_end;
  const void* e_bsrc = ep.bias ? ep.bias : (const void*)w;
  const int e_slot = kv.cache ? kv.slot_map[e_ok ? em : 0] : -1;
  const int e_bidx = (ep.bias && e_ok) ? en : 0;
  const uint32_t e_bias_raw = PBF16 ? (uint32_t)((const bf16_t*)e_bsrc)[e_bidx] : ((const uint32_t*)e_bsrc)[e_bidx];
  da_read_arg(ep.act);
  da_read_arg(ep.out_dtype);
  KvColumn e_col;
  if (kv.cache) e_col = kv_column(kv, en);
  __builtin_amdgcn_sched_barrier(0);                 // the loads stay in this order, ahead of the arithmetic

  // ---- statistics and the normalised rows
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int m = row0 + j * NW;
    if (m >= M) continue;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const int c = (lane + i * 64) * 4;
      sum += (c < K ? 1.f : 0.f) * ((sv[j][i].x + sv[j][i].y) + (sv[j][i].z + sv[j][i].w));
    }
    const float mean = wave_sum(sum) / (float)K * ln.center;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const int c = (lane + i * 64) * 4;
      const float d0 = sv[j][i].x - mean, d1 = sv[j][i].y - mean, d2 = sv[j][i].z - mean, d3 = sv[j][i].w - mean;
      q += (c < K ? 1.f : 0.f) * ((d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3));
    }
    const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)K + ln.eps);
#pragma unroll
    for (int i = 0; i < RV; ++i) {
      const int c = (lane + i * 64) * 4;
      float g4[4], b4[4];
      if (PBF16) {
        g4[0] = __uint_as_float(gq[i].x << 16); g4[1] = __uint_as_float(gq[i].x & 0xffff0000u);
        g4[2] = __uint_as_float(gq[i].y << 16); g4[3] = __uint_as_float(gq[i].y & 0xffff0000u);
        b4[0] = __uint_as_float(bq[i].x << 16); b4[1] = __uint_as_float(bq[i].x & 0xffff0000u);
        b4[2] = __uint_as_float(bq[i].y << 16); b4[3] = __uint_as_float(bq[i].y & 0xffff0000u);
      } else {
        g4[0] = __uint_as_float(gq[i].x); g4[1] = __uint_as_float(gq[i].y); g4[2] = __uint_as_float(gq[i].z); g4[3] = __uint_as_float(gq[i].w);
        b4[0] = __uint_as_float(bq[i].x); b4[1] = __uint_as_float(bq[i].y); b4[2] = __uint_as_float(bq[i].z); b4[3] = __uint_as_float(bq[i].w);
      }
      const float xs[4] = {sv[j][i].x, sv[j][i].y, sv[j][i].z, sv[j][i].w};
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = (xs[e] - mean) * rstd * (g4[e] + ln.gain_offset);
        if (ln.b) y[e] += b4[e];
      }
      uint2 pk = make_uint2((uint32_t)f32_to_bf16(y[0]) | ((uint32_t)f32_to_bf16(y[1]) << 16),
                            (uint32_t)f32_to_bf16(y[2]) | ((uint32_t)f32_to_bf16(y[3]) << 16));
      if (c >= K) pk = make_uint2(0, 0);
      *(uint2*)&a_lds[m][c] = pk;
    }
  }
  // ---- products: a step of w is parked (the first one in front of the barrier: most wavefronts have no row and wait there), then both
  // operands' fragments come out of LDS
  bf16_t* mine = stage[wave];
#pragma unroll
  for (int i = 0; i < WL; ++i) *(uint4*)&mine[(i * 8 + lr) * FL_LD + lc] = wv[0][i];
  lds_barrier();

  floatx4 acc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < SW; ++u) {
    const int k0 = (wave + u * NW) * 64;               // < KMAX: the rows of a are zero from K on
    if (u > 0) {
#pragma unroll
      for (int i = 0; i < WL; ++i) *(uint4*)&mine[(i * 8 + lr) * FL_LD + lc] = wv[u][i];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    if (SW * NW * 64 <= KMAX || k0 < KMAX) {
#pragma unroll
      for (int c = 0; c < 64; c += 32) {
        const bf16x8_t af = __builtin_bit_cast(bf16x8_t, *(const uint4*)&a_lds[fr % AR][k0 + c + fk]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bf16x8_t wf = __builtin_bit_cast(bf16x8_t, *(const uint4*)&mine[(ct * 16 + fr) * FL_LD + c + fk]);
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf, acc[ct], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  }
  if (!APART) lds_barrier();                           // every wavefront is done with its parked steps
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][4 * (lane / 16) + r][ct * 16 + fr] = acc[ct][r];
  lds_barrier();
  if (e_ok) {
    float v = red[0][em][ec];
#pragma unroll
    for (int v2 = 1; v2 < NW; ++v2) v += red[v2][em][ec];
    const float e_bias = !ep.bias ? 0.f : (PBF16 ? __uint_as_float(e_bias_raw << 16) : __uint_as_float(e_bias_raw));
    epilogue_store(ep, em, en, v, e_bias);
    if (kv.cache) kv_column_store(kv, e_col, e_slot, apply_act_bf16(v + e_bias, ep.act));
  }
}

template <int NW, int UN>
static void launch_fused(int mt, dim3 grid, hipStream_t s, const LnPrologue& ln, const bf16_t* W, int ldw,
                         const Epilogue& ep, const KvScatter& kv, int M, int N, int K) {
  if (mt == 1) hipLaunchKernelGGL((gemm_ln_skinny_kernel<1, NW, UN>), grid, dim3(NW * 64), 0, s, ln, W, ldw, ep, kv, M, N, K);
  else hipLaunchKernelGGL((gemm_ln_skinny_kernel<2, NW, UN>), grid, dim3(NW * 64), 0, s, ln, W, ldw, ep, kv, M, N, K);
}

// Up to 8 rows: whether they go to gemm_ln_quads, else to gemm_ln_rows.  By the rows, K and the parameters' dtype, so that a column has the same bits
// among fewer columns; 5 to 8 rows with K from 641 to 1,024 by the columns too.  us, cold weights, recorded one behind the other, gemm_ln_rows / gemm_ln_quads, parameters in bfloat16:
//   1, 4 rows  K =   256, N = 2,304 2.6 / 2.7, 2.6 / 2.7; 6,144 3.2 / 3.0, 3.3 / 3.1
//              K =   768, N = 2,304 3.4 / 3.2, 3.6 / 3.3; 3,072 3.6 / 3.3, 3.7 / 3.4; 8,320 5.1 / 4.8, 5.5 / 4.9; 12,800 5.8 / 5.8, 5.7 / 5.7
//              K = 1,280, N = 4,096 4.8 / 4.9, 4.8 / 5.0; 4,800 5.2 / 5.0, 5.3 / 5.1 (six wavefronts hold up to 1,536; with 32-bit parameters 2 to 9 % behind up
//              to 8,192 columns)
//              K = 1,600, N = 4,800 6.3 / 5.6, 6.6 / 5.6; 6,400 7.3 / 6.9, 7.5 / 6.8; 8,320 9.2 / 7.9, 9.6 / 7.9; 12,800 12.1 / 11.2, 13.1 / 11.0
//   5, 8 rows  every workgroup normalises all rows, here a lane 8 rows' pieces, there a wavefront a row:
//              K =   768, N = 2,304 3.9 / 4.0, 4.1 / 4.1; 8,192 5.6 / 6.9, 5.8 / 6.9; K = 1,536, N = 4,096 5.7 / 6.4, 5.9 / 6.3; 10,240 10.2 / 12.7, 10.9 / 12.8
//              K = 1,600, N = 2,304 - 3 % of the time, 4,096 + 7 %, 4,800 7.4 / 7.2, 7.8 / 7.2; K = 2,048, N = 2,048 6.5 / 5.7, 6.8 / 5.8; 6,144 9.4 / 9.4, 9.9 / 9.3
//              K = 1,024, N = 3,072 4.6 / 4.3, 4,096 + 8 %, 4,800 - 6 %, 6,144 level, 8,192 6.5 / 7.2.  So up to K = 1,024 where its columns a workgroup are 12 or fewer, or
//              17 to 20, for which gemm_ln_rows has two groups of 16.  Recorded steps, all rows / all quads / this: 355M, 5 requests 617 / 611 / 605,
//              8 650 / 645 / 637; 124M, 8 320 / 316 / 318; a Virudra of the 355M's sizes, 5 974 / 958 / 958
static bool ln_quads_takes(int M, int N, int K, int params) {
  if (M > 4) {
    const int share = da_ceil_div(N, 256);
    return M <= 8 && (K > 1536 || (K > 640 && K <= 1024 && (share <= 12 || (share > 16 && share <= 20))));
  }
  return K > 256 && (params == DA_BF16 || K <= 1024 || K > 1280);
}
// Its columns a workgroup, in groups of 4: every compute unit a workgroup up to 8,192 columns, two up to 16,384 as long as they fit side by side; 16 for a
// vocabulary.  With K above 1,024 registers let two workgroups of 28 columns run side by side, with 32-bit parameters of 20: wider ones would run one behind the other,
// and as many as give every compute unit three are ahead.  us, 1 and 4 rows, two a unit / three:
//   bfloat16   N = 14,400, K = 1,600 13.3 / 11.9, 13.1 / 11.7; N = 16,384, K = 1,536 12.4 / 11.8, 12.5 / 11.5; K = 2,048 15.2 / 14.3, 15.1 / 14.1
//              (gemm_ln_rows at N = 16,384: K = 1,032 9.5, where this is 10.4, 1,536 11.4, 1,600 13.3, 2,048 14.7; 4 rows 10.0, 11.7, 14.5, 16.7)
//   32-bit     N = 10,400, K = 1,600 10.5 / 10.1, 10.6 / 10.1; N = 12,800, K = 1,536 10.9 / 10.5, 11.1 / 10.3; K = 2,048 12.5 / 12.2, 12.6 / 12.2; N = 14,336,
//              K = 1,600 12.7 / 11.6, 12.7 / 11.8; beyond three of 20 columns 32 or 16: N = 16,384, K = 1,536 12.5 / 13.8, 12.6 / 14.0, K = 2,048 15.0 / 14.0, 15.1 / 13.8
static int ln_quads_columns(int M, int N, int K, int params) {
  if (N > 64 * 256) return FZ_COLS;
  const int most = params == DA_BF16 ? 28 : 20, two = da_ceil_div(N, 512), three = da_ceil_div(N, 768);
  int share = N <= 32 * 256 ? da_ceil_div(N, 256) : two;
  if (N > 32 * 256 && K > 1024 && M <= 4 && two > most) share = three <= most ? three : (K <= 1536 ? 32 : 16);
  return share <= 16 ? da_ceil_div(share, 4) * 4 : share;
}

// The columns a workgroup of gemm_ln_quads, or 0 where the rows go to another kernel.
extern "C" int da_gemm_bf16_ln_choice(int M, int N, int K, int params) {
  return M > 0 && K <= 2048 && ln_quads_takes(M, N, K, params) ? ln_quads_columns(M, N, K, params) : 0;
}

static int gemm_bf16_norm(const float* x, const int* rows, const void* g, int g_dtype, const void* b,
                          int b_dtype, float eps, float center, float gain_offset, const void* w, int ldw,
                          const void* bias, int bias_dtype, int act, void* out, int out_dtype, int ldo, int M, int N,
                          int K, void* kv_cache, const int* slot_map, int q_cols, int kv_cols, int Hkv, int D, int page,
                          void* stream) {
  DA_REQUIRE(M > 0 && M <= 32 && N > 0 && K > 0, "gemm_bf16_ln: takes 1..32 rows (M=%d N=%d K=%d)", M, N, K);
  DA_REQUIRE(K % 8 == 0 && K <= 256 * FZ_VPL && ldw % 8 == 0 && ldw >= K && ldo >= N,
             "gemm_bf16_ln: K must be a multiple of 8 up to %d (K=%d ldw=%d)", 256 * FZ_VPL, K, ldw);
  DA_REQUIRE(((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0) && ((uintptr_t)g % 16 == 0) &&
             (!b || (uintptr_t)b % 16 == 0), "gemm_bf16_ln: operands must be 16-byte aligned");
  DA_REQUIRE(eps > 0.f, "gemm_bf16_ln: eps must be > 0");
  DA_REQUIRE(act >= DA_ACT_NONE && act <= DA_ACT_LAST, "gemm_bf16_ln: unknown activation %d", act);
  if (kv_cache) {
    DA_REQUIRE(out_dtype == DA_BF16 && q_cols >= 0 && kv_cols == Hkv * D && q_cols + 2 * kv_cols == N && page > 0,
               "gemm_bf16_ln: the q|k|v columns (%d + 2*%d) must add up to N=%d", q_cols, kv_cols, N);
  }
  LnPrologue ln{x, rows, g, g_dtype, b, b_dtype, eps, center, gain_offset};
  Epilogue ep{bias, bias_dtype, act, 0, out, out_dtype, ldo};
  KvScatter kv{kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page};
  dim3 grid(da_ceil_div(N, FZ_COLS));
  const int mt = da_ceil_div(M, 16);
  hipStream_t s = (hipStream_t)stream;
  // Columns a workgroup of gemm_ln_rows: 16 up to 4,096 columns and for a vocabulary; up to 8,192 as many as give every compute unit one
  // workgroup; up to 16,384 as many as give every one two.  16 columns -> this, us:
  //   16 rows, K =   768, N = 8,320 (17, two a unit) 10.0 -> 8.6; N = 12,800 (25) 12.2 -> 9.2
  //    8 rows, K = 1,536, N = 8,200 (17) 10.4 -> 10.0; N = 12,800 14.3 -> 11.9; N = 16,384 (32) 15.0 -> 13.4
  const bool wide = N > 16 * 256 && N <= 64 * 256;
  const int pdt = g_dtype;
  const bool same = (!b || b_dtype == pdt) && (!bias || bias_dtype == pdt) && (pdt == DA_BF16 || pdt == DA_F32);
  const bool quads = same && ln_quads_takes(M, N, K, pdt);
  const bool in_rows = same && !quads && (M <= 8 ? K <= 1536 : M <= 16 && K <= 1024);
  const int cols = quads ? ln_quads_columns(M, N, K, pdt) : (wide ? da_ceil_div(N, N <= 32 * 256 ? 256 : 512) : FZ_COLS);
#define LAUNCH_LN(KERNEL, THREADS)                                                                                 \
  hipLaunchKernelGGL(KERNEL, dim3(da_ceil_div(N, cols)), dim3(THREADS), 0, s, x, rows, g, b, (const bf16_t*)w, ldw, N, K, M | cols << 8, LnRest{eps, center, gain_offset}, ep, kv)
#define LAUNCH_Q(MG, NG, NW, SW)                                                                                   \
  do {                                                                                                            \
    if (pdt == DA_BF16) LAUNCH_LN((gemm_ln_quads_kernel<MG, NG, NW, SW, true>), NW * 64);                          \
    else LAUNCH_LN((gemm_ln_quads_kernel<MG, NG, NW, SW, false>), NW * 64);                                        \
  } while (0)
#define LAUNCH_Q_K(MG, NG)                                                                                         \
  do {                                                                                                            \
    if (MG == 1 && K <= 512) LAUNCH_Q(1, NG, 4, 1);                                                                \
    else if (MG == 1 && K <= 1024) LAUNCH_Q(1, NG, 4, 2);                                                          \
    else if (MG == 1 && K <= 1536) LAUNCH_Q(1, NG, 6, 2);                                                          \
    else LAUNCH_Q(MG, NG, 8, 2);                                                                                   \
  } while (0)
  // (a width more than needed, 4 more columns' loads, takes 1 to 5 % of the launch)
#define LAUNCH_Q_N(MG)                                                                                             \
  do {                                                                                                            \
    switch (da_ceil_div(cols, 4)) {                                                                               \
      case 1: LAUNCH_Q_K(MG, 1); break;                                                                            \
      case 2: LAUNCH_Q_K(MG, 2); break;                                                                            \
      case 3: LAUNCH_Q_K(MG, 3); break;                                                                            \
      case 4: LAUNCH_Q_K(MG, 4); break;                                                                            \
      case 5: LAUNCH_Q_K(MG, 5); break;                                                                            \
      case 6: LAUNCH_Q_K(MG, 6); break;                                                                            \
      case 7: LAUNCH_Q_K(MG, 7); break;                                                                            \
      default: LAUNCH_Q_K(MG, 8); break;                                                                           \
    }                                                                                                             \
  } while (0)
#define LAUNCH_R_P(RV, TWO, CT)                                                                                    \
  do {                                                                                                            \
    if (pdt == DA_BF16) LAUNCH_LN((gemm_ln_rows_kernel<RV, true, TWO, CT>), 512);                                  \
    else LAUNCH_LN((gemm_ln_rows_kernel<RV, false, TWO, CT>), 512);                                                \
  } while (0)
#define LAUNCH_R(RV, TWO)                                                                                          \
  do {                                                                                                            \
    if (cols > 16) LAUNCH_R_P(RV, TWO, 2);                                                                         \
    else LAUNCH_R_P(RV, TWO, 1);                                                                                   \
  } while (0)
  if (quads && M <= 4) LAUNCH_Q_N(1);
  else if (quads && K <= 1024) {                     // (the widths that ln_quads_takes leaves)
    if (cols <= 4) LAUNCH_Q(2, 1, 4, 2);
    else if (cols <= 8) LAUNCH_Q(2, 2, 4, 2);
    else if (cols <= 12) LAUNCH_Q(2, 3, 4, 2);
    else LAUNCH_Q(2, 5, 4, 2);
  } else if (quads) LAUNCH_Q_N(2);
  else if (in_rows && M <= 8) {
    if (K <= 256) LAUNCH_R(1, false);
    else if (K <= 512) LAUNCH_R(2, false);
    else if (K <= 768) LAUNCH_R(3, false);
    else if (K <= 1024) LAUNCH_R(4, false);
    else if (K <= 1280) LAUNCH_R(5, false);
    else LAUNCH_R(6, false);
  } else if (in_rows) {
    if (K <= 256) LAUNCH_R(1, true);
    else if (K <= 512) LAUNCH_R(2, true);
    else if (K <= 768) LAUNCH_R(3, true);
    else LAUNCH_R(4, true);
  } else
    // 8 wavefronts, two chunks in flight each: 125 registers, so two workgroups share a compute unit
    // (deeper unrolling needs 168 and halves that; 16 wavefronts spill)
    launch_fused<8, 2>(mt, grid, s, ln, (const bf16_t*)w, ldw, ep, kv, M, N, K);
  DA_CHECK_LAUNCH("gemm_bf16_ln");
  return 0;
}

extern "C" int da_gemm_bf16_ln(const float* x, const int* rows, const void* g, int g_dtype, const void* b,
                               int b_dtype, float eps, const void* w, int ldw, const void* bias, int bias_dtype,
                               int act, void* out, int out_dtype, int ldo, int M, int N, int K, void* kv_cache,
                               const int* slot_map, int q_cols, int kv_cols, int Hkv, int D, int page,
                               void* stream) {
  return gemm_bf16_norm(x, rows, g, g_dtype, b, b_dtype, eps, 1.0f, 0.0f, w, ldw, bias, bias_dtype, act, out, out_dtype,
                        ldo, M, N, K, kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page, stream);
}

// The same kernels with a root-mean-square norm in front of the product:
//   out = act((x / sqrt(mean(x^2) + eps) * (gain_offset + g)) @ w.T + bias)
extern "C" int da_gemm_bf16_rms(const float* x, const int* rows, const void* g, int g_dtype, float gain_offset,
                                float eps, const void* w, int ldw, const void* bias, int bias_dtype, int act,
                                void* out, int out_dtype, int ldo, int M, int N, int K, void* kv_cache,
                                const int* slot_map, int q_cols, int kv_cols, int Hkv, int D, int page, void* stream) {
  return gemm_bf16_norm(x, rows, g, g_dtype, nullptr, 0, eps, 0.0f, gain_offset, w, ldw, bias, bias_dtype, act, out,
                        out_dtype, ldo, M, N, K, kv_cache, slot_map, q_cols, kv_cols, Hkv, D, page, stream);
}
