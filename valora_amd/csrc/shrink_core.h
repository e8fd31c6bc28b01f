// The direct-load shrink of one tile and one K range, shared by the two-launch shrink kernel and by
// the one-launch decode kernel (which must produce the same bits, chunk for chunk).
//
// One workgroup (4 waves) owns up to 16*MB tokens of one adapter.  Both operands are K-contiguous in
// memory (token rows of x, rank rows of the pool), and v_mfma_f32_16x16x32 wants lane (row = lane%16,
// kgroup = lane/16) to hold 8 consecutive K elements.  Loading that way directly makes neighbouring lanes read
// different rows, and a compute unit then takes some 64 cycles per load instruction, whatever the lines hold: 40 GB/s
// per compute unit measured, against 115-130 GB/s when neighbouring lanes read the same line.  So a wave loads
// blocks of 16 rows x 64 K elements with two instructions of 8 rows x one whole 128-byte line each, and turns a
// block into MFMA operands through a piece of LDS of its own (no barrier, a wave's LDS accesses run in order; 16-byte
// chunks XOR-swizzled by the row so that neither side conflicts).  The four waves take the 64-wide K steps in
// turn, and several steps are requested before any is consumed (the kernel is latency bound: what counts is the
// number of 16-byte loads in flight per lane).
//
// Reference semantics: valora/csrc/bgmv/bgmv_impl.cuh:14-148 (per-token gather mat-vec with the
// rank rows gathered through loc_indicies, fp32 accumulation).
#pragma once

#include <type_traits>

#include "kernel_common.h"

namespace mlora {

constexpr int SHRINK_KSTEP = 64;                      // K elements of a block: one 128-byte line per row
constexpr int SHRINK_BLOCK_BYTES = 16 * SHRINK_KSTEP * 2;
constexpr int SHRINK_STAGE_BLOCKS = 2;                // blocks a wave turns per LDS round trip
constexpr int SHRINK_STAGE_WAVE = SHRINK_STAGE_BLOCKS * SHRINK_BLOCK_BYTES;
// LDS of one tile: the waves' staging pieces, later the four waves' sums
constexpr int shrink_lds_floats(int nblk) {
  return nblk * 4 * 256 > SHRINK_STAGE_WAVE ? nblk * 4 * 256 : SHRINK_STAGE_WAVE;   // (4 pieces / 4 bytes)
}

// four consecutive columns (4*c4 ..) of one token row of the tile shrink_tile_to_lds left in `lds`: the sum of the
// four waves' shares, always in this order
template <int NB, int WAVES = 4>
__device__ __forceinline__ f32x4 shrink_tile_sum(const float *lds, int nblk, int row, int c4) {
  const int b = (row >> 4) * NB + (c4 >> 2);
  const float *src = lds + b * 256 + (row & 3) * 64 + ((row >> 2) & 3) * 16 + (c4 & 3) * 4;
  const f32x4 w0 = *reinterpret_cast<const f32x4 *>(src), w1 = *reinterpret_cast<const f32x4 *>(src + nblk * 256);
  const f32x4 w2 = *reinterpret_cast<const f32x4 *>(src + nblk * 512), w3 = *reinterpret_cast<const f32x4 *>(src + nblk * 768);
  if constexpr (WAVES == 8) {
    const float *const hi = src + nblk * 1024;
    const f32x4 w4 = *reinterpret_cast<const f32x4 *>(hi), w5 = *reinterpret_cast<const f32x4 *>(hi + nblk * 256);
    const f32x4 w6 = *reinterpret_cast<const f32x4 *>(hi + nblk * 512), w7 = *reinterpret_cast<const f32x4 *>(hi + nblk * 768);
    return ((w0 + w4) + (w2 + w6)) + ((w1 + w5) + (w3 + w7));
  }
  return (w0 + w2) + (w1 + w3);
}

// Word 5 of a tile's record on the scalar path (as constant memory: the plan is not written while it is in use; left to itself the
// compiler takes a vector load).
__device__ __forceinline__ int tile_alone(const int32_t *tile) {
  typedef __attribute__((address_space(4))) const int32_t *CP;
  return *(CP)(uintptr_t)(tile + 5);
}

// What a lane without anything to fetch reads, as far as the steps of a batch reach.
__device__ const __align__(128) uint16_t g_shrink_zeros[12 * SHRINK_KSTEP + SHRINK_KSTEP] = {};
constexpr int shrink_steps(int blks) { return blks <= 2 ? 4 : blks <= 5 ? 2 : 1; }
// Leaves the waves' shares of the fp32 result of K range [kbeg, kend) in `lds` (shrink_lds_floats(MB * NB) floats,
// 16-byte aligned), for shrink_tile_sum to add up (rows = tokens of the tile, columns = rank); every thread of the
// workgroup must call it, none may still be reading `lds`, and all have passed a barrier when it returns.
// U: K steps in flight per wave.  The order of the sums does not depend on it.
// until_once (wave-uniform, only looked at with MAY_ONCE): negative where the rows of A have no other reader (shrink_once_tiles).
// Bound by the instructions of one wave in a row, and by what a compute unit takes in.  Rows that are not there are a choice of
// address, not a mask: a mask, four zeroed registers and a branch around each of a batch's 16 loads took 1400 cycles to issue.
// One target, cold layers, masked / like this: 1 token of rank 16 4.9 / 4.0 us, 256 over 64 adapters 6.7 / 5.7, 200 over 16 of rank 32
// 7.6 / 6.5, 77 over ranks 8-64 8.8 / 7.9, 256 over 64 of rank 64 11.6 / 10.9, 512 over 128 of rank 128 29.5 / 28.4.
template <typename T, int MB, int NB, int U = shrink_steps(MB + NB), int WAVES = 4, bool MAY_ONCE = false>
__device__ __forceinline__ void shrink_tile_to_lds(const uint16_t *__restrict__ x, int h_in, const PoolDev &pool,
                                                   int slot, const int32_t *__restrict__ perm, int r, int pos0,
                                                   int cnt, int astart, int kbeg, int kend,
                                                   float *lds, int until_once = 1) {
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int NBLK = MB * NB;
  constexpr int BLKS = MB + NB;                         // 16-row blocks of a K step, x first
  constexpr bool MANY = NB > 2;
  constexpr bool PINNED = MB == 1 && NB > 4;
  constexpr bool WHOLE = MB == 1 || NB <= 2;            // has a loop of its own for whole batches
  static_assert(WAVES * (U - 1) <= 12, "a batch's steps reach past g_shrink_zeros");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, kg = lane >> 4;           // MFMA operand roles
  const int grow = lane >> 3, gcol = lane & 7;          // loader roles: row within a group of 8, 16-byte chunk
  const int64_t base = (int64_t)astart + (int64_t)r * slot;
  if (MAY_ONCE) asm volatile("" : "+s"(until_once));   // (requested with the rest, not in front of the first batch)

  // This lane's row pointers (already at its chunk).  All look-ups are requested together, one round trip: those with
  // nothing to look up read an address that is always there instead of branching around the load.
  const bool indexed = pool.a_loc_len > 0;
  const int64_t *const a_loc = indexed ? pool.a_loc : reinterpret_cast<const int64_t *>(perm);
  int tok[MB][2];
  int64_t prow[NB][2];
  bool ok[NB][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int row = mb * 16 + u * 8 + grow;
      tok[mb][u] = perm[pos0 + (row < cnt ? row : 0)];   // (a row past the tile's end reads the first one's)
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int j = nb * 16 + u * 8 + grow;
      // (up to rank 32 a row past the rank reads the last one, its results are never used; above, where whole blocks may
      // be missing, it reads zeros that stay in the cache)
      const int64_t idx = base + (MANY ? j : min(j, r - 1));
      ok[nb][u] = indexed && (!MANY || j < r) && idx >= 0 && idx < pool.a_loc_len;
      prow[nb][u] = a_loc[ok[nb][u] ? idx : 0];
    }
  }
  const uint16_t *rp[BLKS][2];
  int step[NB][2];          // MANY: all bits where the row moves on with K, none where it stays on its zeros
  bool all = true;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) rp[mb][u] = x + (uint64_t)(uint32_t)tok[mb][u] * (uint32_t)h_in + gcol * 8;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      ok[nb][u] = ok[nb][u] && prow[nb][u] >= 0 && prow[nb][u] < pool.w_rows;
      all = all && ok[nb][u];
      rp[MB + nb][u] = pool.w + (uint64_t)(uint32_t)(ok[nb][u] ? prow[nb][u] : 0) * (uint32_t)h_in + gcol * 8;
      step[nb][u] = ok[nb][u] ? -1 : 0;
      // (PINNED: kept in its register, not as a condition in two scalar ones, of which there are none left: 46 and more stood in lanes of
      // vector registers.  512 tokens of rank 128 on one adapter, a pass 242 / 238 us)
      if (PINNED) asm("" : "+v"(step[nb][u]));
      if (MANY && !ok[nb][u]) rp[MB + nb][u] = as_global(g_shrink_zeros) + gcol * 8;
    }
  }
  // Whole batches can be loaded as they are: rows that are not there read zeros anyway, or there are none.
  // (Tiles of several token blocks above rank 32 go without: the addresses of both loops at once spill.  32 tokens, rank 64, 13
  // registers spilled / without that loop: 600 tokens over 16 adapters 7.1 / 6.8 us, 1152 over 64 13.9 / 12.7, 3000 over 32 17.5 / 16.1,
  // 4000 over 128 23.4 / 22.6.)
  const bool plain = WHOLE && (MANY || __builtin_amdgcn_ballot_w64(!all) == 0ull);

  // where this lane's chunks sit in a staged block: row u*8 + grow / chunk gcol when it writes what it loaded,
  // row lrow / chunk 4*c + kg when it reads operand c (K elements c*32 + kg*8 .. + 8 of the step)
  unsigned char *const mine = reinterpret_cast<unsigned char *>(lds) + wave * SHRINK_STAGE_WAVE;
  unsigned char *const wptr = mine + grow * 128 + ((gcol ^ grow) << 4);       // + u * 1024: the row's low bits stay
  const unsigned char *rptr[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) rptr[c] = mine + lrow * 128 + (((c * 4 + kg) ^ (lrow & 7)) << 4);

  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 buf[U * BLKS][2];
  auto use = [&]() {
#pragma unroll
    for (int b0 = 0; b0 < U * BLKS; b0 += SHRINK_STAGE_BLOCKS) {
#pragma unroll
      for (int b = b0; b < b0 + SHRINK_STAGE_BLOCKS && b < U * BLKS; ++b)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          *reinterpret_cast<u32x4 *>(wptr + (b - b0) * SHRINK_BLOCK_BYTES + u * 1024) = buf[b][u];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int b = b0; b < b0 + SHRINK_STAGE_BLOCKS && b < U * BLKS; ++b)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          buf[b][c] = *reinterpret_cast<const u32x4 *>(rptr[c] + (b - b0) * SHRINK_BLOCK_BYTES);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // a K step's x blocks come before its A blocks, so both operands of these products are there
#pragma unroll
      for (int b = b0; b < b0 + SHRINK_STAGE_BLOCKS && b < U * BLKS; ++b) {
        const int uu = b / BLKS, nb = b % BLKS - MB;
        if (nb == 0 || (nb > 0 && nb * 16 < r)) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
              acc[mb][nb < 0 ? 0 : nb] = Tr::mfma(as<vec8>(buf[uu * BLKS + mb][c]), as<vec8>(buf[b][c]), acc[mb][nb < 0 ? 0 : nb]);
        }
      }
    }
  };
  // The trip counts must be wave-uniform: MFMA ignores EXEC, so a lane that left a loop early would still feed its stale
  // registers into the matrix core.
  // Whole batches: a load is an instruction, the steps of a batch are offsets in it.  (A loop for either kind of A: with a branch in one
  // loop 900 tokens of rank 128 on one adapter take 277 us a pass, with two 269.)
  int kb0 = kbeg + wave * SHRINK_KSTEP;
  auto whole_batches = [&](auto a_once) {
    for (; plain && kb0 + (WAVES * (U - 1) + 1) * SHRINK_KSTEP <= kend; kb0 += WAVES * SHRINK_KSTEP * U) {
#pragma unroll
      for (int b = 0; b < BLKS; ++b)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint16_t *const src = rp[b][u] + (MANY && b >= MB ? kb0 & step[b < MB ? 0 : b - MB][u] : kb0);
          if (decltype(a_once)::value && b >= MB) {
#pragma unroll
            for (int uu = 0; uu < U; ++uu) buf[uu * BLKS + b][u] = load16_once(src + uu * WAVES * SHRINK_KSTEP);
          } else {
#pragma unroll
            for (int uu = 0; uu < U; ++uu) buf[uu * BLKS + b][u] = load16(src + uu * WAVES * SHRINK_KSTEP);
          }
        }
      requested();
      use();
    }
  };
  if (MAY_ONCE && until_once < 0) whole_batches(std::true_type{});
  else whole_batches(std::false_type{});
  // what is left of the chunk, less than a batch (or all of it, where a rank row lies outside the index or the pool): steps and
  // lanes past its end read zeros, and so do rows that are not there
  for (; kb0 < kend; kb0 += WAVES * SHRINK_KSTEP * U) {
#pragma unroll
    for (int uu = 0; uu < U; ++uu) {
      const int k = kb0 + uu * WAVES * SHRINK_KSTEP;
      const bool kok = k + gcol * 8 < kend;
#pragma unroll
      for (int b = 0; b < BLKS; ++b)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int nb = b < MB ? 0 : b - MB;
          buf[uu * BLKS + b][u] = load16(as_global(kok && (b < MB || (PINNED ? step[nb][u] != 0 : ok[nb][u])) ? rp[b][u] + k : g_shrink_zeros));
        }
    }
    requested();
    use();
    if (MANY && WHOLE) break;   // (it is less than a batch)
  }

  // Every wave leaves its share as it is (C layout: column = lane%16, rows = 4*(lane/16)+i) and whoever needs an
  // element adds the four up: two barriers, where a tree of the waves takes four and idles most of them.
  __syncthreads();   // the staging pieces are done with
  float *const dst = lds + wave * NBLK * 256;
#pragma unroll
  for (int b = 0; b < NBLK; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[(b * 4 + i) * 64 + lane] = acc[b / NB][b % NB][i];
  __syncthreads();
}

// From how many tiles of the list on A is read as lines that nobody reads again (load16_once), by a tile that is its adapter's only one;
// shrink_kernel, 16-token tiles.  The record says whether it is, and of how many: the host knows the resident adapters, not those that a
// batch touches, and where tiles share A such loads lose most (512 tokens of rank 128 on one of 128 adapters, a pass 243 us without, 299 with
// them; 900 of rank 32 on four 354 / 385).  From 4 MB of A on, more than an L2 holds (one token over 8 adapters, a pass of 64 calls
// 379 / 398); in rows of whole lines; above rank 16, up to which the look at the flag takes 0.12 us of a launch of 5 and the loads give no more
// (256 tokens over 64 adapters of rank 16, a pass of 256 one-call launches 1518 us plain, 1536 with them; rank 8 alone 0.993); and not for
// batches of five tokens a tile and more.  A pass, plain loads / this: 512 tokens over 128 adapters of rank 128
// 633 / 611 us, 900 over 128 of rank 64 563 / 537, 77 over ranks 8-64 473 / 456; twelve batches of 14 to 900 tokens 1.026 in the mean, and
// twelve of as many tokens on one to four of up to 128 adapters 1.00 to 1.09 (what is above 1.02 is y written through)
// (the one-launch op, which has no scalar register left for it, reads A the plain way: 256 tokens over 64 adapters of rank 16, a pass
// of 16 layers 453 us, 450 with such loads).
inline int shrink_once_tiles(const ShrinkArgs &a, int64_t n_tiles, int max_rank) {
  const int64_t tile_bytes = (int64_t)a.rp * a.h_in * a.n_targets * 2;
  if (max_rank <= 16 || a.compensate || a.T >= 5 * n_tiles || (a.h_in & 63) || (reinterpret_cast<uintptr_t>(a.pool.w) & 127u)) return 0x7fffffff;
  return (int)((((int64_t)4 << 20) + tile_bytes - 1) / tile_bytes);
}

}  // namespace mlora
