// The tile height of the plans that the one-call entry points cut for themselves (csrc/api.hip, csrc/binding.cpp).
#pragma once
#include <cstdint>

namespace mlora {

// Tokens a workgroup where the shrink of a one-call entry point is faster with all of K in one workgroup (shrink_whole_kernel)
// than with the table's tiles and split, else 0.  (Not for planned ops: their results must not depend on how many targets they
// are given, nor on the tile height.)  It is while 32-token pieces, or 64-token ones up to rank 16, run in one round of a
// workgroup per compute unit, x is most of what such a workgroup reads, and K not too long.  The shrink alone, cold x, the
// table's tiles / this, us:
//   4096 wide: 5000 tokens over 8 adapters, rank 8 13.9 / 11.7, rank 16 14.9 / 12.3 (rank 64 17.2 / 19.4; 5600 over 32, rank 32
//   17.1 / 18.2); 7000 over 32, rank 16 17.1 / 14.4, rank 32 22.9 / 17.4 (over 100, more than one round, rank 32 26.9 / 27.1);
//   14000 over 32, rank 16, 64 a workgroup 28.3 / 24.9 (rank 32 31.4 / 31.1); 3500 over 8, rank 8 9.6 / 10.7
//   5000 over 32: 5120 wide, rank 16 19.6 / 15.6, 3072 wide, rank 16 12.9 / 10.2 (8192 wide, rank 16 23.1 / 23.8)
//   2048 wide, rank 64: 6700 over 64 19.9 / 14.8 (10000 over 32, rank 32 by 64 a workgroup 15.0 / 17.3)
// Through the entry points, 180 shapes of 4500 to 15500 tokens, 2048 to 5120 wide: 0.93 in the mean.  Values that are not the rounded
// exact sum: 0.138 / 0.124 %.
inline int one_call_tile(int64_t T, int64_t A, int64_t max_rank, int64_t h_in) {
  if (T < 4480 || max_rank > 64 || h_in > 5120 || h_in * max_rank > 131072) return 0;
  const int64_t tails = (A < T ? A : T) / 2;   // an adapter's last piece is half empty in the mean
  const int64_t by32 = T / 32 + tails, by64 = T / 64 + tails;
  if (by32 <= 256) return max_rank > 16 && h_in > 3072 && by32 < 192 ? 0 : 32;
  return max_rank <= 16 && by64 >= 160 && by64 <= 256 ? 64 : 0;
}

}  // namespace mlora
