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
// and a width of 1,024, by 10 to 15 % of a decode step; up to 8 rows (which take half the LDS, so that the
// workgroups still run side by side) up to a width of 2,048.  Every workgroup reads and normalises all rows again (at a
// width of 1,600 that is 2.5 us of vector work a compute unit), so beyond a width of 1,536, where no two workgroups of more
// than 16 columns fit on a compute unit, and beyond 8,192 columns, which are three and four rounds of 16, the norm is
// a kernel of its own from 5 rows on: us, fused / two kernels, 5 and 8 rows, K = 1,600: N = 8,200 11.3 / 10.4 and 12.1 / 10.6, 12,800 14.5 / 13.4
// and 15.9 / 13.7; K = 1,920, N = 10,240 13.0 / 12.3 and 14.5 / 12.7 (3 rows 11.1 / 12.3); but K = 2,048, where the product takes 12 wavefronts, N = 10,240
// 13.4 / 14.4 and 14.9 / 14.8.  Never for a vocabulary.
extern "C" int da_can_fuse_ln(int n_rows, int K, int N) {
  const bool fits = (n_rows <= 16 && K <= 1024) || (n_rows <= 8 && K <= 2048);
  const bool slower = n_rows > 4 && K > 1536 && K < 2048 && N > 8192;
  return n_rows > 0 && fits && !slower && K % 8 == 0 && N <= 16384;
}
