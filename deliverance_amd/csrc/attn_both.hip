// Attention of a step that holds both one-token sequences and portions of prompts, in one launch: the workgroups of
// attn_prefill.hip (4 row blocks x 2 key phases) and those of attn_decode.hip (8 wavefronts a pair), both of 512 threads, side by
// side.  Launched one behind the other, a portion of a few hundred rows leaves most compute units without a workgroup
// for as long as its longest one walks its keys, and the decode rows wait for that.  The portions' workgroups come first: they
// are the long ones.  Each row's sums are those of its own kernel in that form.
// Measured on MI355X, us, the two kernels one behind the other / this one: 16 heads, 40 sequences of 600 keys beside 512 rows after 256
// keys 32.2 / 22.3, beside 64 rows 26.9 / 21.6; 8 sequences beside 512 rows 20.8 / 14.2; 60 of 1,000 keys beside 512 rows 54.5 / 43.6;
// 25 heads, 60 of 900 keys 80.3 / 72.9; 12 heads, 3 sequences of 100 keys beside 20 rows after 500 19.8 / 11.7.
#define DA_ATTN_BODIES 1
#include "attn_decode.hip"
#include "attn_prefill.hip"

// (157 registers, as the prefill form needs them: one workgroup a compute unit.  Held to 128, two decode workgroups fit, but the portions
// spill: the first of the above 24.6, 8 sequences beside 512 rows 18.0, 60 of 1,000 keys 41.6)
template <bool BT_LDS>
__global__ void __launch_bounds__(512, 2)
attn_both_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache, const int* __restrict__ block_table,
                 const int* __restrict__ seq_lens, int n_portions, int n_blocks, int Hq, int q_ld, int max_blocks, int Hkv,
                 const int* __restrict__ q_start, int n_decode, int page, float scale, int window, bf16_t* __restrict__ out, int out_ld) {
  const int pairs = n_portions * Hq, id = (int)blockIdx.x - pairs * n_blocks;
  if (id < 0) {
    const int pair = (int)blockIdx.x % pairs;
    attn_prefill_body<4, 4, 2, BT_LDS, false>(pair / Hq, pair % Hq, (int)blockIdx.x / pairs, n_blocks, q, cache, block_table, q_start, seq_lens, q_ld,
                                       max_blocks, Hq, Hkv, n_decode, page, scale, window, out, out_ld);
    return;
  }
  attn_decode_body<2, 8, false>(id / Hq, id % Hq, q, cache, block_table, seq_lens, q_ld, max_blocks, Hq, Hkv, 64, page, scale, window, out, out_ld, 0, nullptr);
}

// 1 for the steps that this kernel takes: both kinds of sequences, heads of 64, contexts whose pairs are not shared out, and
// portions that leave compute units idle (128-row workgroups no more than compute units).
extern "C" int da_attn_both_takes(int n_decode, int n_portions, int max_query_len, int Hq, int D, int page, int splits) {
  if (n_decode <= 0 || n_portions <= 0 || D != 64 || splits > 1 || !(page == 8 || page == 16 || page == 32 || page == 64)) return 0;
  return (long)da_ceil_div(max_query_len, 128) * Hq * n_portions <= PF_PHASED_MAX_WORKGROUPS && (long)n_decode * Hq < (1L << 30);
}

// 1 when a step's attention goes to this kernel.  It holds one workgroup a compute unit where the decode kernel holds two, and its
// portions have 4 row blocks x 2 key phases whatever their length.  us, the two kernels / this one:
//  - many pairs of one-token rows, which want that second workgroup: 1,024 pairs of 20 keys beside 15 rows 13.0 / 13.3, of 300 21.6 / 18.6;
//    1,575 of 50 beside 2 rows 16.6 / 17.0, beside 16 rows 20.9 / 17.4; 1,536 of 20 beside 16 rows of a table of 16 keys 15.4 / 17.2, beside five
//    times 512 rows 32.0 / 33.8; 2,048 of 50 beside 256 rows 20.7 / 21.6, of 300 32.1 / 32.6; 3,060 and more 10 to 40 % behind up to 300 keys (of
//    1,000: 119 / 114).  So up to 1,024 pairs, or 1,600 beside 16 rows or more, if the block tables are wider than 256 keys and the
//    portions' workgroups at most 128;
//  - portions of up to 64 rows after many keys, which the prefill kernel gives four key phases: 360 pairs of 20 keys beside 16 rows
//    after 500 keys 16.8 / 13.0, after 1,000 21.3 / 17.2, after 1,900 28.9 / 27.2 (32 rows 28.6 / 28.8), after 4,000 42.4 / 51.4, after
//    8,000 77 / 96.  So up to 1,920 keys by the block table's width; longer portions have the same form in both.
extern "C" int da_attn_both_pays(int n_decode, int n_portions, int max_query_len, int Hq, int D, int page, int splits, int max_blocks) {
  if (!da_attn_both_takes(n_decode, n_portions, max_query_len, Hq, D, page, splits)) return 0;
  const long pairs = (long)n_decode * Hq;
  const long keys = (long)max_blocks * page, portions = (long)da_ceil_div(max_query_len, 128) * Hq * n_portions;
  const bool more = max_query_len >= 16 && keys > 256 && portions <= 128;
  return pairs <= (more ? 1600 : 1024) && (max_query_len > 64 || keys <= 1920);
}

// The first n_decode sequences bring one row each (row s is sequence s's), the n_portions behind them the rows q_start says.
extern "C" int da_attn_both(const void* q, int q_ld, const void* cache, const int* block_table, int max_blocks, const int* q_start,
                            const int* seq_lens, int n_decode, int n_portions, int max_query_len, int Hq, int Hkv, int D, int page,
                            float scale, int window, void* out, int out_ld, void* stream) {
  DA_REQUIRE(Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && max_query_len > 0, "attn_both: bad sizes (%d and %d heads, %d rows)", Hq, Hkv, max_query_len);
  DA_REQUIRE(da_attn_both_takes(n_decode, n_portions, max_query_len, Hq, D, page, 1), "attn_both: %d one-token sequences and %d portions of up to %d rows, head size %d",
             n_decode, n_portions, max_query_len, D);
  DA_REQUIRE(q_ld >= Hq * D && out_ld >= Hq * D && q_ld % 8 == 0 && out_ld % 4 == 0, "attn_both: row lengths");
  DA_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)cache % 16 == 0 && (uintptr_t)out % 8 == 0, "attn_both: operands must be 16-byte aligned");
  DA_REQUIRE(window >= 0 && max_blocks > 0 && scale > 0.f, "attn_both: bad window, block table or scale");
  const int n_blocks = da_ceil_div(max_query_len, 128);
  const dim3 grid(n_portions * Hq * n_blocks + n_decode * Hq);
#define AB_GO(L) hipLaunchKernelGGL((attn_both_kernel<L>), grid, dim3(512), 0, (hipStream_t)stream, (const bf16_t*)q, (const bf16_t*)cache, \
                                    block_table, seq_lens, n_portions, n_blocks, Hq, q_ld, max_blocks, Hkv, q_start, n_decode, page, scale, window, \
                                    (bf16_t*)out, out_ld)
  if (max_blocks <= PF_BT_MAX_PHASED) AB_GO(true); else AB_GO(false);
#undef AB_GO
  DA_CHECK_LAUNCH("attn_both");
  return 0;
}
