// Products into the residual stream whose k is shared out over workgroups: the kernels of gemm_skinny32.h and gemm_wide.hip, each share's
// sums in rows of their own, and the rules of when.  (A unit of its own: in gemm_mfma.hip's library the kernels beside them, instruction
// for instruction the same, lay elsewhere, and a Virudra's recorded step took 1,109 us for 1,099.)
#include "gemm_skinny32.h"

// How many shares the k of a product into the residual stream can be cut into (1: none; da_gemm_bf16 adds into the stream).  With few
// tiles and a long K most compute units have no tile; cut, share by share, they have one, and what the shares' sums cost is
// that the norm behind reads them (da_layernorm_join; never a norm that is fused into its product: more rows than
// da_can_fuse_ln takes).  Whole slabs of 64 k, 8 shares at most; the last share may be shorter than the others, which have 512 k and more.
//  - up to 64 rows (32 columns a workgroup, gemm_skinny32), K from 4,096, more than 1,024 columns: us, cold weights, += / shares: 64
//    rows, N = 1,600, K = 6,400 14.1 / 10.2 (5), 32 rows 11.1 / 8.0, 16 rows 10.3 / 7.9.  Not N = 1,024, K = 4,096: 64 rows 7.4 / 6.5, 48 rows
//    7.5 / 5.9, but with 8 shares for the norm to read a step of 64 rows takes 1,249 us for 1,232; nor N = 768, K = 3,072 (64 rows 4.9 / 5.5);
//  - more rows: tiles of 128 x 128 where they are at most 85, as many shares as bring them to about 256 (552 rows, N = 1,024,
//    K = 4,096 20.1 / 12.2 (6)).  K from 2,048.  (K = 1,024: 552 rows 7.5 / 6.5, which the norm's reads take up; so do they
//    with two shares of more rows: 1,624 rows, K = 4,096 29.7 / 23.9, a step of them 2,834 / 2,841.)
struct GemmShares { int shares, k_share, shape; };     // shape: DA_WIDE_..., or DA_WIDE_NONE for gemm_skinny32
static GemmShares gemm_shares(int M, int N, int K) {
  const GemmShares none{1, K, DA_WIDE_NONE};
  if (M <= 8 || (M <= 64 && N <= 1024) || N % 4 || K % 64 || N > 2048) return none;
  GemmShares g = none;
  long tiles;
  if (M <= 64) {
    if (K < 4096) return none;
    tiles = da_ceil_div(N, 32);
  } else {
    if (K < 2048) return none;
    tiles = (long)da_ceil_div(M, 128) * da_ceil_div(N, 128);
    if (tiles > 85) return none;
    g.shape = DA_WIDE_128x128;
  }
  long n = 256 / tiles;
  if (n > K / 512) n = K / 512;
  if (n > 8) n = 8;
  if (n < 2) return none;
  g.k_share = da_ceil_div(K / 64, n) * 64;
  g.shares = da_ceil_div(K, g.k_share);
  return g;
}
extern "C" int da_gemm_shares(int M, int N, int K) { return M > 0 && N > 0 && K > 0 ? gemm_shares(M, N, K).shares : 1; }

// How many shares a step cuts it into: as many, where a layer with its norm is faster by them.  Measured as whole steps of 12 layers, us
// a layer gained (all of K = 4 N but where said):
//  - up to 64 rows: K = 6,400 16 rows 0.0, 24 and 32 -0.6, 33 0.3, 48 and 64 1.6; K = 5,120 16 rows 0.4, 33 -1.2, 48 -0.1, 49 0.6, 64 1.0 (and,
//    product and norm alone, N = 2,048, K = 4,096 -0.8 to -1.0 from 24 to 64 rows): from 33 rows with K from 6,144, from 49 with K from 5,120;
//  - more rows: 2 to 18 up to 840 rows (K = 4,096 0.9 at 400, -0.9 to 1.5 from 552 to 700); above, K = 2,048 -0.4 from 1,100 rows, K = 3,072 -0.6
//    at 900, -2.5 at 1,100, -2.4 at 1,300, K = 4,096 -1.3 at 900, -1.6 at 1,024, but 5.3 at 1,100, K = 5,120 10 and more.  With a shorter K
//    (product and norm alone): N = 1,024, K = 2,048 0.5 at 400 rows, -0.6 at 552, -3.7 at 1,024; N = 2,048, K = 4,096 1.6 at 256, -1.1 at 400 (64
//    tiles), 6.9 at 552 (80).
extern "C" int da_gemm_step_shares(int M, int N, int K) {
  const int n = da_gemm_shares(M, N, K);
  if (n == 1) return 1;
  bool pays;
  if (M <= 64) pays = (M > 32 && K >= 6144) || (M > 48 && K >= 5120);
  else {
    const bool many = M > 840 && ((N >= 512 && K < 4096) || (N >= 1024 && K < 5120 && M <= 1024));
    const bool short_k = K < 3 * N && M > 384 && (long)da_ceil_div(M, 128) * da_ceil_div(N, 128) <= 64;
    pays = !many && !short_k;
  }
  return pays ? n : 1;
}

// partial[s] = a @ w.T over share s of k, [M, N] each, 32-bit; as many shares as da_gemm_shares says (more than one).
extern "C" int da_gemm_bf16_shares(const void* a, int lda, const void* w, int ldw, float* partial, int M, int N, int K, void* stream) {
  DA_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_bf16_shares: bad sizes M=%d N=%d K=%d", M, N, K);
  DA_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && lda >= K && ldw >= K, "gemm_bf16_shares: lda and ldw must be multiples of 8 and hold K (K=%d lda=%d ldw=%d)", K, lda, ldw);
  DA_REQUIRE((uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0, "gemm_bf16_shares: operands must be 16-byte aligned");
  if (M == 0) return 0;
  const GemmShares g = gemm_shares(M, N, K);
  DA_REQUIRE(g.shares > 1, "gemm_bf16_shares: a product of %d rows, N=%d, K=%d is not shared out", M, N, K);
  DA_REQUIRE(partial && (uintptr_t)partial % 16 == 0, "gemm_bf16_shares: the sums' place must be 16-byte aligned");
  const Epilogue ep{nullptr, 0, DA_ACT_NONE, 0, partial, DA_F32, N};
  const KvScatter kv{nullptr, nullptr, 0, 0, 0, 0, 0};
  hipStream_t s = (hipStream_t)stream;
  const bf16_t *A = (const bf16_t*)a, *W = (const bf16_t*)w;
  if (g.shape != DA_WIDE_NONE) da_gemm_wide_launch(s, A, lda, W, ldw, ep, kv, M, N, K, g.shape, g.k_share);
  else {
    DA_REQUIRE(lda <= (1 << 24) && ldw <= (1 << 24), "gemm_bf16_shares: rows lie too far apart (lda=%d ldw=%d)", lda, ldw);
    const dim3 grid(da_ceil_div(N, 32), g.shares);
#define DA_SK32_GO(AL, P) hipLaunchKernelGGL((gemm_skinny32_kernel<AL, 8, P, true>), grid, dim3(512), 0, s, A, W, ep.out, lda, ldw, ep.ldo, M, N, K, 32, g.k_share, ep.bias, epilogue_rest(ep), kv)
    if (M <= 16) DA_SK32_GO(2, 4);
    else if (M <= 32) DA_SK32_GO(4, 3);
    else if (M <= 48) DA_SK32_GO(6, 2);
    else DA_SK32_GO(8, 2);
#undef DA_SK32_GO
  }
  DA_CHECK_LAUNCH("gemm_bf16_shares");
  return 0;
}
