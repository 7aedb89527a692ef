// Which kernel form a step of a given shape takes, where the host and the layer loop of run_step.hip must agree.
#include "common.h"

// Decode attention splits a (sequence, head) pair's keys over workgroups when the pairs alone leave most
// of the chip idle and the context is long: shares of at least 1,024 keys, as many as bring the
// workgroups to about 512, 32 at most.  The choice reads the step's shape only (pairs and the width of
// the block table), so that a recorded step keeps it.
extern "C" int da_decode_splits(int n_seqs, int n_heads, int max_blocks, int page) {
  const long by_keys = ((long)max_blocks * page) / 1024;
  const long pairs = (long)n_seqs * n_heads;
  const long by_fill = 512 / (pairs > 0 ? pairs : 1);
  long n = by_keys < by_fill ? by_keys : by_fill;
  if (n > 32) n = 32;
  return n >= 2 ? (int)n : 1;
}

// Measured on MI355X inside the model: the fused norm + product kernel wins up to 16 rows (one row tile)
// and a width of 1,024, by 10 to 15 % of a decode step; up to 8 rows up to a width of 2,048.  Every workgroup reads and normalises all rows again, so with
// 5 rows and more, beyond a width of 1,536 and about 5,000 columns, the norm is a kernel of its own.  us, fused / two kernels, cold weights, recorded one behind
// the other, 5 and 8 rows: K = 1,600, N = 4,800 7.2 / 8.0, 7.2 / 8.0; N = 6,400 8.5 / 7.7, 8.6 / 7.7; N = 8,192 10.0 / 8.7, 10.1 / 8.9; N = 12,800 16.8 / 12.7,
// 17.1 / 13.2; K = 1,920, N = 7,680 10.4 / 9.7, 10.5 / 10.1; K = 2,048, where the product takes 12 wavefronts, N = 6,144 9.2 / 9.6, 9.3 / 9.9; N = 8,192 10.6 / 10.4,
// 10.8 / 10.6; N = 10,240 14.0 / 13.6, 14.4 / 13.7 (K = 1,536, N = 10,240 10.2 / 11.5, 10.9 / 11.7; 4 rows, K = 1,600, N = 12,800 10.4 / 12.8).  Never for a
// vocabulary.
extern "C" int da_can_fuse_ln(int n_rows, int K, int N) {
  const bool fits = (n_rows <= 16 && K <= 1024) || (n_rows <= 8 && K <= 2048);
  const bool slower = n_rows > 4 && K > 1536 && N > (K < 1920 ? 5120 : 6144);
  return n_rows > 0 && fits && !slower && K % 8 == 0 && N <= 16384;
}
