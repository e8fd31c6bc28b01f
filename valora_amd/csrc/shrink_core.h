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
template <int NB>
__device__ __forceinline__ f32x4 shrink_tile_sum(const float *lds, int nblk, int row, int c4) {
  const int b = (row >> 4) * NB + (c4 >> 2);
  const float *src = lds + b * 256 + (row & 3) * 64 + ((row >> 2) & 3) * 16 + (c4 & 3) * 4;
  const f32x4 w0 = *reinterpret_cast<const f32x4 *>(src), w1 = *reinterpret_cast<const f32x4 *>(src + nblk * 256);
  const f32x4 w2 = *reinterpret_cast<const f32x4 *>(src + nblk * 512), w3 = *reinterpret_cast<const f32x4 *>(src + nblk * 768);
  return (w0 + w2) + (w1 + w3);
}

// Leaves the four waves' shares of the fp32 result of K range [kbeg, kend) in `lds` (shrink_lds_floats(MB * NB) floats,
// 16-byte aligned), for shrink_tile_sum to add up (rows = tokens of the tile, columns = rank); every thread of the
// workgroup must call it, none may still be reading `lds`, and all have passed a barrier when it returns.
// U: K steps in flight per wave.  The order of the sums does not depend on it.
constexpr int shrink_steps(int blks) { return blks <= 2 ? 4 : blks <= 5 ? 2 : 1; }
template <typename T, int MB, int NB, int U = shrink_steps(MB + NB)>
__device__ __forceinline__ void shrink_tile_to_lds(const uint16_t *__restrict__ x, int h_in, const PoolDev &pool,
                                                   int slot, const int32_t *__restrict__ perm, int r, int pos0,
                                                   int cnt, int astart, int kbeg, int kend,
                                                   float *lds) {
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int NBLK = MB * NB;
  constexpr int BLKS = MB + NB;                         // 16-row blocks of a K step, x first
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, kg = lane >> 4;           // MFMA operand roles
  const int grow = lane >> 3, gcol = lane & 7;          // loader roles: row within a group of 8, 16-byte chunk
  const int64_t base = (int64_t)astart + (int64_t)r * slot;

  // This lane's row pointers (already at its chunk).  All look-ups are requested together, one round trip: those with
  // nothing to look up read an address that is always there instead of branching around the load.
  const bool indexed = pool.a_loc_len > 0;
  const int64_t *const a_loc = indexed ? pool.a_loc : reinterpret_cast<const int64_t *>(perm);
  int tok[MB][2];
  int64_t prow[NB][2];
  bool ok[BLKS][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int row = mb * 16 + u * 8 + grow;
      ok[mb][u] = row < cnt;
      tok[mb][u] = perm[pos0 + (row < cnt ? row : 0)];
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int j = nb * 16 + u * 8 + grow;
      const int64_t idx = base + j;
      ok[MB + nb][u] = indexed && j < r && idx >= 0 && idx < pool.a_loc_len;
      prow[nb][u] = a_loc[ok[MB + nb][u] ? idx : 0];
    }
  }
  const uint16_t *rp[BLKS][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) rp[mb][u] = x + (int64_t)tok[mb][u] * h_in + gcol * 8;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      ok[MB + nb][u] = ok[MB + nb][u] && prow[nb][u] >= 0 && prow[nb][u] < pool.w_rows;
      rp[MB + nb][u] = pool.w + (ok[MB + nb][u] ? prow[nb][u] : 0) * h_in + gcol * 8;
    }
  }

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

  // The trip count must be wave-uniform: MFMA ignores EXEC, so a lane that left the loop early
  // would still feed its stale registers into the matrix core.  Lanes past the end load zeros.
  for (int kb0 = kbeg + wave * SHRINK_KSTEP; kb0 < kend; kb0 += 4 * SHRINK_KSTEP * U) {
    u32x4 buf[U * BLKS][2];
#pragma unroll
    for (int uu = 0; uu < U; ++uu) {
      const int k = kb0 + uu * 4 * SHRINK_KSTEP;
      const bool kok = k + gcol * 8 < kend;
#pragma unroll
      for (int b = 0; b < BLKS; ++b)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          buf[uu * BLKS + b][u] = (ok[b][u] && kok) ? load16(rp[b][u] + k) : u32x4{0, 0, 0, 0};
    }
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
        if (nb >= 0 && nb * 16 < r) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
              acc[mb][nb < 0 ? 0 : nb] = Tr::mfma(as<vec8>(buf[uu * BLKS + mb][c]), as<vec8>(buf[b][c]), acc[mb][nb < 0 ? 0 : nb]);
        }
      }
    }
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

}  // namespace mlora
