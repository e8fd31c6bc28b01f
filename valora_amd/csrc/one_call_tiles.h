// The tile height of the plans that the one-call entry points cut for themselves (csrc/api.hip, csrc/binding.cpp).
#pragma once
#include <cstdint>

namespace mlora {

// Tokens a workgroup where the shrink of a one-call entry point is faster with all of K in one workgroup (shrink_whole_kernel)
// than with the table's tiles and split, else 0.  (Planned ops keep the plan's tiles and split: for one plan their results do not
// depend on the number of targets, nor on the height among 16, 32 and 64 tokens.)  It is while 32-token pieces, or 64-token ones up
// to rank 16, run in one round of a workgroup per compute unit, x is most of what such a workgroup reads, and K not too long.  How
// many pieces there are depends on how many of the index's adapters the batch touches, which the host does not know: the least
// (all tokens of one adapter) must be enough of them where few lose, and the usual number, half a piece more for every adapter,
// with some room for tails, not too many.
// The shrink alone, cold x, the table's tiles / this, us:
//   4096 wide: 5000 tokens over 8 adapters, rank 8 13.9 / 11.7, rank 16 14.9 / 12.3 (rank 64 17.2 / 19.4; 5600 over 32, rank 32
//   17.1 / 18.2); 7000 over 32, rank 16 17.1 / 14.4, rank 32 22.9 / 17.4 (over 100, more than one round, rank 32 26.9 / 27.1; 6119 over 2,
//   rank 32 18.5 / 20.2); 14000 over 32, rank 16, 64 a workgroup 28.3 / 24.9 (rank 32 31.4 / 31.1); 3500 over 8, rank 8 9.6 / 10.7
//   5000 over 32: 5120 wide, rank 16 19.6 / 15.6, 3072 wide, rank 16 12.9 / 10.2 (8192 wide, rank 16 23.1 / 23.8)
//   2048 wide, rank 64: 6700 over 64 19.9 / 14.8 (10000 over 32, rank 32 by 64 a workgroup 15.0 / 17.3); 2560 wide, rank 32: 7554 over one
//   adapter 15.4 / 15.9, batches of more than ten adapters 0.86 in the mean
//   64 a workgroup: 7186 over 42 of 168, rank 8, 3072 wide, 127 workgroups 16.1 / 19.4; 15521 over 19, rank 16, 2560 wide, 258 21.8 / 27.6
// Through the entry points, 1500 shapes of 4480 to 17000 tokens, 1024 to 5120 wide, batches of one to all of up to 220 adapters: 0.90 in
// the mean of the 1113 that it takes, 14 above 1.02.  Values that are not the rounded exact sum: 0.138 / 0.124 %.
inline int one_call_tile(int64_t T, int64_t A, int64_t max_rank, int64_t h_in) {
  if (T < 4480 || max_rank > 64 || h_in > 5120 || h_in * max_rank > 131072) return 0;
  const int64_t touched = A < T ? A : T, least32 = (T + 31) / 32, least64 = (T + 63) / 64;
  const int64_t tails = touched / 2 + (touched < 12 ? touched : 12) / 2;   // (the second term: room for more than the mean)
  if (least32 + tails <= 256) {
    if (max_rank <= 16 || h_in <= 2048) return 32;
    if (h_in < 3072) return A >= 8 ? 32 : 0;
    return h_in <= 3072 || least32 >= 200 ? 32 : 0;
  }
  return max_rank <= 16 && h_in >= 3072 && least64 >= 140 && least64 + tails <= 256 ? 64 : 0;
}

}  // namespace mlora
