// LoRA shrink for gfx950:  v[row, j] = T( sum_k x[t, k] * A_a[j, k] )
//
// shrink_kernel: one workgroup (4 waves) owns one adapter-grouped tile of up to 16*MB tokens and one K chunk
// (shrink_core.h has the loads and the products).  Bound by its chain of round trips, not by bytes: tile record ->
// look-ups -> operand loads -> cross-wave sum -> hand-over of the K chunks (what it measured is in shrink_core.h).
// shrink_whole_kernel: the same with all of K in one workgroup of eight waves, for one-call entry points.
// shrink_gemm_kernel: 128- and 256-token tiles, one target of rank up to 64.  shrink_targets_kernel: 128-token tiles, several
// targets together, or one above rank 64.
//
// Split-K without atomics on values: every workgroup writes its fp32 partial tile; the chunks are summed in index order
// (bit-reproducible) by the last chunk of a small tile to arrive, by shrink_reduce_kernel or by the expand.
//
// Reference semantics: valora/csrc/bgmv/bgmv_impl.cuh:14-148 (per-token gather mat-vec with the
// rank rows gathered through loc_indicies, fp32 accumulation, one T store per output).
#include <type_traits>

#include "kernel_common.h"
#include "shrink_core.h"

namespace mlora {

namespace {


// the arguments of target z of a multi-target launch
__device__ __forceinline__ ShrinkArgs select_target(const ShrinkArgs &a, int z) {
  ShrinkArgs p = a;
  p.slot = a.slots[z];
  p.out = a.out + (int64_t)z * a.out_tstride;
  p.partial = a.partial + (int64_t)z * a.partial_tstride;
  return p;
}

// A compensation call (csrc/api.hip, mlora_lora_compensate) multiplies the tokens of a plan by two adapters: each
// token's own, tile by tile as always, and as a second "target" the one that is merged into the base weights.  The
// second needs no tile list: its tiles are runs of `bm` positions, whatever adapters their tokens have.
// (The kernels take the flag from a leading argument, beside reduce_here: a load of the argument block in front of the
// tile's look-ups cost every shrink launch 0.2 us.)
constexpr int SHRINK_COMPENSATE = 4;
__device__ __forceinline__ void merged_tile(const int32_t *plan, int tile_idx, int bm, int &r, int &pos0, int &cnt, int &astart) {
  r = plan[H_MERGED_RANK];
  astart = plan[H_MERGED_START];
  pos0 = tile_idx * bm;
  cnt = r > 0 ? min(bm, plan[H_NACTIVE] - pos0) : 0;
}

template <typename T>
__device__ __forceinline__ void store_v(const ShrinkArgs &p, int pos, int t, int r, int col, float v) {
  using Tr = Traits<T>;
  if (p.out_by_token) {
    // the caller's matrix, one row per token (dispatch_bgmv and friends)
    uint16_t *dst = p.out + (int64_t)t * p.out_stride + col;
    if (col < r && col < p.ncols) {
      if (p.mode == MLORA_SHRINK_ACCUMULATE) v += Tr::to_float(*dst);
      *dst = Tr::from_float(v);
    } else if (p.mode == MLORA_SHRINK_ZERO_PAD && col < p.width) {
      *dst = 0;
    }
  } else {
    // internal v buffer, one row of rp columns per sorted position; columns >= r hold zero
    if (col < p.rp) p.out[(int64_t)pos * p.out_stride + col] = Tr::from_float(col < r ? v : 0.f);
  }
}

// four consecutive columns at once: one 8-byte store where they all hold values and the row allows it
template <typename T>
__device__ __forceinline__ void store_v4(const ShrinkArgs &p, int pos, int t, int r, int c4, f32x4 v) {
  using Tr = Traits<T>;
  const int col = 4 * c4;
  uint16_t *dst = p.out + (int64_t)(p.out_by_token ? t : pos) * p.out_stride + col;
  const bool whole = p.out_by_token ? col < r && col + 4 <= p.ncols && p.mode != MLORA_SHRINK_ACCUMULATE &&
                                          (reinterpret_cast<uintptr_t>(dst) & 7u) == 0
                                    : col < p.rp;
  if (whole) {
    if (col >= r) v = f32x4{0.f, 0.f, 0.f, 0.f};   // ranks are multiples of 8
    *reinterpret_cast<uint2 *>(dst) = uint2{Tr::pack2(v[0], v[1]), Tr::pack2(v[2], v[3])};
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) store_v<T>(p, pos, t, r, col + i, v[i]);
}

// v[row, :] = T(sum_s partial[s][row][:]) for every row that has an adapter; one thread per four columns, a workgroup the rows
// that fit whole (partial rows stand one after the other: a thread's offset in the workgroup's piece is its index).
// Bound by a launch and three round trips (arguments, chunks, store): a few MB.  Four or eight chunks are requested before any
// is used, beside the row's look-ups; no division.  With 64-bit divisions, a round trip per conditional chunk and 2-byte stores:
// 7600 tokens of rank 32 in four chunks 3.5 us a launch, now 2.7.
// ONCE: the chunks are read as lines that nobody reads again (launch_shrink_reduce).
template <typename T, bool ONCE>
__global__ __launch_bounds__(256) void shrink_reduce_kernel(const int32_t *h_plan, const float *h_partial, int h_quarter, float h_inv_quarter,
                                                            int h_flags, int h_ksplit, ShrinkArgs args_in) {
  const ShrinkArgs p = select_target(args_in, blockIdx.y);
  const bool merged = (h_flags & SHRINK_COMPENSATE) && blockIdx.y == 1;
  const int rows = 256 / h_quarter, tid = threadIdx.x;
  const int row = (int)(((float)tid + 0.5f) * h_inv_quarter), c4 = tid - row * h_quarter;   // exact: tid < 256
  const int pos0 = (int)blockIdx.x * rows;
  const bool on = row < rows && pos0 + row < p.T;      // others read the piece's first element and store nothing
  const int pos = pos0 + (on ? row : 0);
  const char *chunk = as_global(reinterpret_cast<const char *>(h_partial)) + ((int64_t)blockIdx.y * p.partial_tstride + (int64_t)pos0 * h_quarter * 4) * 4;
  const uint32_t at = on ? (uint32_t)tid * 16u : 0u;
  const int64_t stride = (int64_t)p.T * h_quarter * 16;
  const int32_t *__restrict__ plan = as_global(h_plan);
  const int n_active = plan[H_NACTIVE], merged_rank = plan[H_MERGED_RANK];
  // (a compensation leaves most positions out: what it would read for them costs more than to wait for the count first; 6246
  // tokens of rank 128, most of them with the merged adapter, a pass of 14 layers 4530 us, so 4349)
  if ((h_flags & SHRINK_COMPENSATE) && pos0 >= n_active) return;
  const int own_rank = (plan + p.off_prank)[pos], tok = (plan + p.off_perm)[pos];
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  auto add_chunks = [&](auto batch, int s0) {
    constexpr int BATCH = decltype(batch)::value;
    f32x4 q[BATCH];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const f32x4 *const src = reinterpret_cast<const f32x4 *>(chunk + at);
      if constexpr (ONCE) q[u] = __builtin_nontemporal_load(src);
      else q[u] = *src;
      chunk = next_chunk(chunk, s0 + u + 1 < h_ksplit, stride);
    }
    requested();
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
      if (s0 + u < h_ksplit) v += q[u];   // wave-uniform
  };
  if (h_ksplit <= 4) add_chunks(std::integral_constant<int, 4>{}, 0);
  else
    for (int s0 = 0; s0 < h_ksplit; s0 += 8) add_chunks(std::integral_constant<int, 8>{}, s0);
  const int r = merged ? merged_rank : own_rank;
  if (on && pos < n_active && r > 0) store_v4<T>(p, pos, tok, r, c4, v);   // (no rank: nothing was computed for the token)
}

// The leading scalar parameters repeat what the first dependent load (the tile record) needs: with kernel-argument
// preloading they arrive in registers at launch, so that load does not wait for a load of the argument block.
// Waves per SIMD the register allocator has to leave room for: as many as do without spills.  (Three for 64-token tiles up to rank 32
// spill 4 and 28 registers; three / two: 4000 tokens over 32 adapters of rank 32, four chunks 12.8 / 11.6 us, eight 12.9 / 11.4; 8000 over
// 64 of rank 16 18.4 / 16.0, of rank 32 20.6 / 18.7.)
constexpr int shrink_min_waves(int mb, int nb) { return mb + nb <= 3 ? 4 : nb == 8 ? 3 - mb : mb == 4 ? 2 : 3; }
// ONCE: a tile that is its adapter's only one may read A as lines that nobody reads again (shrink_once_tiles), above rank 16.  A form of its own: with both
// loops in one kernel a call of a few tokens takes 3.78 us instead of 3.62.
template <typename T, int MB, int NB, bool ONCE>
__global__ __launch_bounds__(256, shrink_min_waves(MB, NB)) void shrink_kernel(const int32_t *tiles_base, int h_ksplit, int h_n_targets, int h_reduce_here,
                                                     int h_n_tiles, ShrinkArgs args_in) {
  int tile_idx, z_idx, s;
  const bool compensate = (h_reduce_here & SHRINK_COMPENSATE) != 0;
  const int reduce_here = h_reduce_here & ~SHRINK_COMPENSATE;
  if (reduce_here) {
    // The K chunks of a tile are summed by whichever of them finishes last, out of the L2 they share: the id mod 8
    // selects the XCD, so all chunks (and targets) of a tile get ids that agree mod 8: grid (8 tiles x chunks, targets, 8 tiles).
    s = (int)blockIdx.x >> 3;
    z_idx = (int)blockIdx.y;
    tile_idx = (int)blockIdx.z * 8 + ((int)blockIdx.x & 7);
    if (tile_idx >= h_n_tiles) return;
  } else {
    // workgroup id = (tile * targets + target) * ksplit + K chunk.  The id mod 8 selects the XCD, so
    // with the K chunk as the fast index the tiles of an adapter that share a K chunk of A, and the
    // targets that share a K chunk of x, meet in one L2.
    const int wg_tz = blockIdx.x / h_ksplit;
    tile_idx = wg_tz / h_n_targets;
    z_idx = wg_tz - tile_idx * h_n_targets;
    s = blockIdx.x - wg_tz * h_ksplit;
  }
  const int32_t *__restrict__ tile = tiles_base + (int64_t)tile_idx * TILE_WORDS;
  const ShrinkArgs p = select_target(args_in, z_idx);
  constexpr int NBLK = MB * NB;
  constexpr int QUARTER = NB * 4;                        // groups of four columns per row, a power of two
  constexpr int ITEMS = (MB * 16 * QUARTER + 255) / 256; // (row, group) pairs per thread
  __shared__ __align__(16) float s_tile[shrink_lds_floats(NBLK)];
  __shared__ int s_last;

  int r = tile[1], pos0 = tile[2], cnt = tile[3], astart = tile[4];
  const int until_once = ONCE ? p.once_tiles - 1 - tile_alone(tile) : 1;
  if (compensate && z_idx == 1) merged_tile(p.plan, tile_idx, 16 * MB, r, pos0, cnt, astart);
  if (cnt <= 0) return;   // records past the last tile are zero
  const int32_t *__restrict__ perm = p.plan + p.off_perm;
  const int kbeg = s * p.kchunk;
  const int kend = min(p.h_in, kbeg + p.kchunk);
  const int tid = threadIdx.x;
  const int quarter = p.rp >> 2;                         // rp is a multiple of 16, at most NB * 16
  // thread -> (row, group of four columns); the token of the row where the result goes to token order
  bool on[ITEMS];
  int row[ITEMS], c4[ITEMS], tok[ITEMS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int e = tid + it * 256;
    row[it] = e / QUARTER;
    c4[it] = e & (QUARTER - 1);
    on[it] = row[it] < cnt && c4[it] < quarter;
    tok[it] = (p.out_by_token && on[it]) ? perm[pos0 + row[it]] : 0;
  }
  shrink_tile_to_lds<T, MB, NB, shrink_steps(MB + NB), 4, ONCE>(p.x, p.h_in, p.pool, p.slot, perm, r, pos0, cnt, astart, kbeg, kend, s_tile, until_once);
  if (p.ksplit == 1) {
#pragma unroll
    for (int it = 0; it < ITEMS; ++it)
      if (on[it]) store_v4<T>(p, pos0 + row[it], tok[it], r, c4[it], shrink_tile_sum<NB>(s_tile, NBLK, row[it], c4[it]));
    return;
  }
  // this K chunk's fp32 partial (ordinary stores).  Where the chunks are not summed here, a later launch on the
  // stream does it -- shrink_reduce_kernel, or the expand itself for small batches -- in index order, rounding once.
  const uint32_t pq = (uint32_t)(reduce_here ? p.prp >> 2 : quarter);
  const int64_t sstride = (int64_t)p.T * pq * 16;         // bytes between chunks
  char *const part = as_global(reinterpret_cast<char *>(p.partial)) + (int64_t)pos0 * pq * 16;
  uint32_t at[ITEMS];                                    // of the thread's items, lanes without one on the first
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) at[it] = on[it] ? ((uint32_t)row[it] * pq + (uint32_t)c4[it]) * 16u : 0u;
#pragma unroll
  for (int it = 0; it < ITEMS; ++it)
    if (on[it]) *reinterpret_cast<f32x4 *>(part + s * sstride + at[it]) = shrink_tile_sum<NB>(s_tile, NBLK, row[it], c4[it]);
  if (!reduce_here) return;

  // ---- split-K summed here: every chunk leaves its partial in the L2, the last one to arrive adds them up.
  // Partials are plain stores into rows that own whole 128-byte lines (prp floats per row), so a line never
  // holds rows of two tiles and no compute unit has read it before the tile is complete.  A chunk announces
  // itself -- after its stores have been acknowledged by the L2 -- by adding to the tile's arrival word (one
  // atomic per workgroup, device scope): the count in the low byte, and one more count in the field of the XCD
  // it runs on.  Whoever brings the count to ksplit is the last: it knows all partials are written, and from
  // its XCD's field whether all of them were written through ITS L2.  If so it reads them back (L2 hits) and
  // sums them in index order; if not (the workgroups of the tile were not placed the way the id layout
  // expects) it computes every chunk itself, in the same order with the same code: same bits, no waiting
  // anywhere, and nothing depends on where or when a workgroup runs.  It then puts the word back to zero for
  // the next launch on this plan (launches that share a plan must not overlap).
  // (Worth it for small tiles only: one workgroup reads ksplit x tile x prp x 4 bytes at L2 latency.  For
  // 128-token tiles of rank 64 that is 256 KB and measured 8.5 us, against 3.7 us for the reduce launch.)
  // (With one item a thread and 64 of them, wave 0 holds them all: the others only wait for its verdict.)
  constexpr bool ONE_WAVE = NBLK == 1;
  wait_vmcnt<0>();
  if (!ONE_WAVE) __syncthreads();
  int last = 0;
  if (!ONE_WAVE || tid < 64) {
    if (tid == 0) {
      const uint32_t xcd = xcd_id();
      unsigned long long *word = p.arrive + (int64_t)tile_idx * MLORA_MAX_TARGETS + z_idx;
      const unsigned long long add = 1ull + (xcd < 8 ? 1ull << (8 + 7 * xcd) : 0ull);
      const unsigned long long now = __hip_atomic_fetch_add(word, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
      if ((int)(now & 0xffull) == p.ksplit) {
        const bool all_here = xcd < 8 && (int)((now >> (8 + 7 * xcd)) & 0x7full) == p.ksplit;
        last = (all_here && reduce_here == 1) ? 1 : 2;
        __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      s_last = last;
    }
  }
  __syncthreads();
  last = s_last;
  if (last == 0) return;
  f32x4 v[ITEMS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) v[it] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (last == 1) {
    if (ONE_WAVE && tid >= 64) return;
    // v[row, :] = T(0 + p_0 + p_1 + ...): the order shrink_reduce_kernel uses.  The loads of a batch of chunks are
    // requested for all of the thread's items together (the last chunk again where there are fewer).
    auto add_chunks = [&](auto batch) {
      constexpr int BATCH = decltype(batch)::value;
      const char *chunk = part;
      for (int s0 = 0; s0 < p.ksplit; s0 += BATCH) {
        f32x4 q[ITEMS][BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
#pragma unroll
          for (int it = 0; it < ITEMS; ++it) q[it][u] = *reinterpret_cast<const f32x4 *>(chunk + at[it]);
          chunk = next_chunk(chunk, s0 + u + 1 < p.ksplit, sstride);
        }
        requested();
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
          if (s0 + u < p.ksplit) {   // wave-uniform
#pragma unroll
            for (int it = 0; it < ITEMS; ++it) v[it] += q[it][u];
          }
      }
    };
    if (ITEMS > 2 || p.ksplit <= 4) add_chunks(std::integral_constant<int, 4>{});
    else add_chunks(std::integral_constant<int, ITEMS <= 2 ? 8 : 4>{});
  } else {
    // the chunks were not all written through this XCD's L2 (or the caller asked for this path): compute them
    // here, one after the other.  (The empty asm keeps the compiler from computing this path's addresses early and
    // holding them through the ordinary one.)
    int pos_r = pos0, astart_r = astart;
    asm volatile("" : "+s"(pos_r), "+s"(astart_r));
    for (int c = 0; c < p.ksplit; ++c) {
      const int kb = c * p.kchunk;
      __syncthreads();   // everybody has read the previous chunk's sums
      shrink_tile_to_lds<T, MB, NB, 1>(p.x, p.h_in, p.pool, p.slot, perm, r, pos_r, cnt, astart_r, kb,
                                       min(p.h_in, kb + p.kchunk), s_tile);
#pragma unroll
      for (int it = 0; it < ITEMS; ++it)
        if (on[it]) v[it] += shrink_tile_sum<NB>(s_tile, NBLK, row[it], c4[it]);
    }
  }
#pragma unroll
  for (int it = 0; it < ITEMS; ++it)
    if (on[it]) store_v4<T>(p, pos0 + row[it], tok[it], r, c4[it], v[it]);
}

// All of K in one workgroup of eight waves, 32 or 64 tokens: no partials, no second launch (or wait for the other chunks).  The
// tile list may be one of taller tiles, whose pieces of 16 * MB tokens the workgroups take.  csrc/one_call_tiles.h has the rule.
// Bound by launch, look-ups, first loads and the final sums, which nothing hides with one workgroup a compute unit (130 registers at rank
// 32), and between them by what a compute unit takes in: 7000 tokens over 32 adapters, 4096 wide, rank 32 read 57 MB in 17.4 us,
// 3.3 TB/s over the whole launch.  The shrink alone, cold x, 128-token tiles in four chunks and the launch that sums them / this: rank 32 22.9 / 17.4 us,
// rank 16 17.1 / 14.4; four waves instead of eight with the same 32 tokens 19.6 / 16.4 (6749 tokens, rank 32).  Four K steps in
// flight a wave instead of two gain nothing at 4096 and lose where they leave a remainder (7000 tokens, 3072 wide, rank 8
// 10.8 / 12.1).
constexpr int WHOLE_WAVES = 8;
constexpr int WHOLE_RUN = 4;   // consecutive pieces that run on one XCD
constexpr int whole_lds_floats(int nblk) {
  return nblk * WHOLE_WAVES * 256 * 4 > WHOLE_WAVES * SHRINK_STAGE_WAVE ? nblk * WHOLE_WAVES * 256 : WHOLE_WAVES * SHRINK_STAGE_WAVE / 4;
}
template <typename T, int MB, int NB>
__global__ __launch_bounds__(512, 2) void shrink_whole_kernel(const int32_t *tiles_base, int h_n_pieces, int h_pieces, ShrinkArgs p) {
  // The workgroup id mod 8 selects the XCD: a run of WHOLE_RUN pieces, most of them one adapter's, meets there.
  constexpr int H = 16 * MB;
  const int id = (int)blockIdx.x;   // (one target)
  const int piece = (id / (8 * WHOLE_RUN)) * (8 * WHOLE_RUN) + (id & 7) * WHOLE_RUN + (id >> 3) % WHOLE_RUN;
  if (piece >= h_n_pieces) return;
  const int tile_idx = piece >> h_pieces, from = (piece - (tile_idx << h_pieces)) * H;   // 1 << h_pieces pieces a tile
  const int32_t *__restrict__ tile = tiles_base + (int64_t)tile_idx * TILE_WORDS;
  constexpr int NBLK = MB * NB, QUARTER = NB * 4;        // groups of four columns per row, a power of two
  __shared__ __align__(16) float s_tile[whole_lds_floats(NBLK)];
  int r = tile[1], pos0 = tile[2], cnt = tile[3], astart = tile[4];
  pos0 += from;
  cnt = min(cnt - from, H);
  if (cnt <= 0) return;   // records past the last tile are zero
  const int32_t *__restrict__ perm = p.plan + p.off_perm;
  shrink_tile_to_lds<T, MB, NB, MB + NB <= 5 ? 2 : 1, WHOLE_WAVES>(p.x, p.h_in, p.pool, p.slot, perm, r, pos0, cnt, astart, 0, p.h_in, s_tile);
  const int quarter = p.rp >> 2;
#pragma unroll 1
  for (int e = threadIdx.x; e < cnt * QUARTER; e += 64 * WHOLE_WAVES) {
    const int row = e / QUARTER, c4 = e & (QUARTER - 1);
    if (c4 < quarter)
      store_v4<T>(p, pos0 + row, p.out_by_token ? perm[pos0 + row] : 0, r, c4, shrink_tile_sum<NB, WHOLE_WAVES>(s_tile, NBLK, row, c4));
  }
}

// What a rank row that is not there reads, K step after K step (one 128-byte line).
__device__ const __align__(128) uint16_t g_zero_line[64] = {};

// Prefill-sized tiles (128 or 256 tokens): a GEMM tile.  The four waves split the tile's tokens, so no cross-wave reduction
// is needed.  A K step of 64 is requested into registers as whole 128-byte lines, every wave its own x rows and a quarter
// of the adapter's A rows, two steps before it is used, and handed over through two LDS stages; one barrier per step.
//
// Bound by a fixed part (launch, look-ups, first step, partials: one step only takes 6.6 of 17.9 us; 5254 tokens of rank 64, one target in
// four chunks, 16.7 since x is read once and partials are written through, launch_shrink) and then by a stream of loads at 4.3 TB/s: 43 MB
// of x, and A again per 128 tokens from L2.  Of the 17.9 us, 17.1 with the loads alone, 12.3 with the products alone; a deeper ring, K starts
// spread over the channels, ids by XCD and contiguous pool rows change nothing.  Direct global -> LDS loads into a three-stage ring (one or two workgroups a compute unit instead of three, LDS turn
// of the result, zero rows read for a narrower adapter's rank) / now, behind the same expand: three targets of 5254 tokens of
// rank 64 37.2 / 33.4 us, 5401 tokens over ranks 8-64, one target 20.4 / 19.6, two 29.5 / 25.6, three 34.5 / 30.7, `down` of 11008
// 56.6 / 54.9 (targets together: shrink_targets_kernel, below).  (The chunks summed inside the launch by the last to arrive: 20.4
// against 15.3 + 5.1 for the two launches, and 43 against 34 + 5 for three targets of rank 64.)
constexpr int GEMM_KC = 64;                             // K elements of a step: one 128-byte line per row
constexpr int gemm_stage_bytes(int nb, int mbw) { return (64 * mbw + 16 * nb) * GEMM_KC * 2; }
constexpr int GEMM_AHEAD = 2;                           // steps requested before the first is used

// Two 16-column blocks of a token row's fp32 partial, as the products leave them (four columns a lane, `row` the same for four lanes),
// written through to memory (store16_through): the lanes of a pair, two rows, exchange a block first, so that a store writes whole
// lines.  at: column 4 * kg of the first block in row `row & ~1`, `rp` floats in front of the next row's.  All lanes take part.
__device__ __forceinline__ void store_partials_through(float *at, int rp, const f32x4 &first, const f32x4 &second, int row, int cnt, bool odd) {
  const u32x4 lo = as<u32x4>(first), hi = as<u32x4>(second), give = odd ? lo : hi;
  u32x4 got;
#pragma unroll
  for (int i = 0; i < 4; ++i) got[i] = lane_pair(give[i]);
  uint16_t *const dst = reinterpret_cast<uint16_t *>(at + (odd ? 16 : 0));
  if ((row & ~1) < cnt) store16_through(dst, odd ? got : lo);
  if ((row | 1) < cnt) store16_through(dst + 2 * rp, odd ? hi : got);
}

// One tile and one K chunk, NB 16-row blocks of rank (of the tile's own adapter), MBW 16-token blocks per wave.  ONCE: the rows of x have
// no other reader (launch_shrink).
template <typename T, int NB, int MBW, bool ONCE>
__device__ __forceinline__ void shrink_gemm_tile(const ShrinkArgs &p, int s, int r, int pos0, int cnt, int astart, unsigned char *lds) {
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int KC = GEMM_KC, KS = KC / 32;
  constexpr int XG = MBW * 2;                           // 8-row groups (1 KB) of x per wave and step
  constexpr int AG = NB * 2;                            // 8-row groups of A per step, shared
  constexpr int APW = AG >= 4 ? AG / 4 : 1;             // of which a wave loads
  constexpr int STAGE = gemm_stage_bytes(NB, MBW);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, kg = lane >> 4;           // MFMA operand roles
  const int grow = lane >> 3, gcol = lane & 7;          // loader roles: row within an 8-row group, 16-byte chunk
  const int32_t *__restrict__ perm = as_global(p.plan) + p.off_perm;
  const int64_t base = (int64_t)astart + (int64_t)r * p.slot;
  const int wrow0 = wave * 16 * MBW;

  // this lane's global row pointers (already at its chunk), all look-ups in one round trip: a row past the tile's end reads the
  // first one's, a rank row that is not there a line of zeros on which it stays
  const bool indexed = p.pool.a_loc_len > 0;
  const int64_t *const a_loc = indexed ? as_global(p.pool.a_loc) : reinterpret_cast<const int64_t *>(perm);
  int tok[XG];
  int64_t prow[APW];
  bool ok[APW];
#pragma unroll
  for (int g = 0; g < XG; ++g) {
    const int row = wrow0 + g * 8 + grow;
    tok[g] = perm[pos0 + (row < cnt ? row : 0)];
  }
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    const int j = (wave * APW + i) % AG * 8 + grow;     // (rank 16 has two groups: they are loaded and written twice)
    const int64_t idx = base + j;
    ok[i] = indexed && j < r && idx >= 0 && idx < p.pool.a_loc_len;
    prow[i] = a_loc[ok[i] ? idx : 0];
  }
  const uint16_t *xp[XG], *ap[APW];
  int astep[APW];                                       // all bits: the row moves on with K; none: it stays on its line
  const uint16_t *const zeros = as_global(g_zero_line) + gcol * 8;
#pragma unroll
  for (int g = 0; g < XG; ++g) xp[g] = as_global(p.x) + (uint64_t)(uint32_t)tok[g] * (uint32_t)p.h_in + gcol * 8;
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    ok[i] = ok[i] && prow[i] >= 0 && prow[i] < p.pool.w_rows;
    ap[i] = ok[i] ? as_global(p.pool.w) + (uint64_t)(uint32_t)prow[i] * (uint32_t)p.h_in + gcol * 8 : zeros;
    astep[i] = ok[i] ? -1 : 0;
  }

  const int kbeg = s * p.kchunk;
  const int kend = min(p.h_in, kbeg + p.kchunk);
  const int n_steps = (kend - kbeg) / KC;               // whole ones
  u32x4 rx[GEMM_AHEAD][XG], ra[GEMM_AHEAD][APW];
  auto request = [&](int step, u32x4 (&x)[XG], u32x4 (&a)[APW]) {
    const int off = kbeg + step * KC;
#pragma unroll
    for (int g = 0; g < XG; ++g) x[g] = ONCE ? load16_once(xp[g] + off) : load16(xp[g] + off);
#pragma unroll
    for (int i = 0; i < APW; ++i) a[i] = load16(ap[i] + (off & astep[i]));
    requested();
  };
  // Row R of a stage (x rows of the four waves, then A) stands at R * 128, its chunk c at chunk c ^ (R & 7): 8 lanes write one
  // row, and the 16 rows of an MFMA operand spread over the banks.
  unsigned char *const wx = lds + (wrow0 + grow) * 128 + ((gcol ^ grow) << 4);
  unsigned char *const wa = lds + (64 * MBW + wave * APW % AG * 8 + grow) * 128 + ((gcol ^ grow) << 4);
  const unsigned char *rxp[KS], *rap[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    rxp[ks] = lds + (wrow0 + lrow) * 128 + (((ks * 4 + kg) ^ (lrow & 7)) << 4);
    rap[ks] = lds + (64 * MBW + lrow) * 128 + (((ks * 4 + kg) ^ (lrow & 7)) << 4);
  }

  f32x4 acc[MBW][NB];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto put = [&](int stage, const u32x4 (&x)[XG], const u32x4 (&a)[APW]) {
#pragma unroll
    for (int g = 0; g < XG; ++g) *reinterpret_cast<u32x4 *>(wx + stage + g * 1024) = x[g];
#pragma unroll
    for (int i = 0; i < APW; ++i) *reinterpret_cast<u32x4 *>(wa + stage + i * 1024) = a[i];
    requested();
  };
  auto multiply = [&](int stage) {
    // behind this barrier the stage is complete, and everybody has read the other one
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
    requested();
    u32x4 xf[KS][MBW], bf[KS][NB];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int mb = 0; mb < MBW; ++mb) xf[ks][mb] = *reinterpret_cast<const u32x4 *>(rxp[ks] + stage + mb * 2048);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) bf[ks][nb] = *reinterpret_cast<const u32x4 *>(rap[ks] + stage + nb * 2048);
    }
    if (MBW * NB <= 8) requested();   // (all operands of a step requested together)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb) acc[mb][nb] = Tr::mfma(as<vec8>(bf[ks][nb]), as<vec8>(xf[ks][mb]), acc[mb][nb]);
    requested();
  };
  // (the loop's requests, and those in front of it, under no condition: the compiler has to know how many are outstanding
  // where it waits)
  int step = 0;
  if (n_steps >= 2 * GEMM_AHEAD) {
#pragma unroll
    for (int i = 0; i < GEMM_AHEAD; ++i) request(i, rx[i], ra[i]);
    do {
#pragma unroll
      for (int i = 0; i < GEMM_AHEAD; ++i) {
        put(((step + i) & 1) * STAGE, rx[i], ra[i]);
        request(step + i + GEMM_AHEAD, rx[i], ra[i]);
        multiply(((step + i) & 1) * STAGE);
      }
      step += GEMM_AHEAD;
    } while (step + 2 * GEMM_AHEAD <= n_steps);
  } else {
#pragma unroll
    for (int i = 0; i < GEMM_AHEAD; ++i)
      if (i < n_steps) request(i, rx[i], ra[i]);
  }
#pragma unroll
  for (int i = 0; i < 2 * GEMM_AHEAD - 1; ++i)
    if (step + i < n_steps) {
      put(((step + i) & 1) * STAGE, rx[i % GEMM_AHEAD], ra[i % GEMM_AHEAD]);
      if (i < GEMM_AHEAD && step + i + GEMM_AHEAD < n_steps) request(step + i + GEMM_AHEAD, rx[i % GEMM_AHEAD], ra[i % GEMM_AHEAD]);
      multiply(((step + i) & 1) * STAGE);
    }
  const int off = kbeg + n_steps * KC;
  if (off < kend) {   // the end of a K that is not a multiple of 64: chunks past it read zeros
    const bool kok = off + gcol * 8 < kend;
#pragma unroll
    for (int g = 0; g < XG; ++g) rx[0][g] = load16(as_global(kok ? xp[g] + off : zeros));
#pragma unroll
    for (int i = 0; i < APW; ++i) ra[0][i] = load16(as_global(kok && astep[i] ? ap[i] + off : zeros));
    put((n_steps & 1) * STAGE, rx[0], ra[0]);
    multiply((n_steps & 1) * STAGE);
  }
  // A lane has four consecutive rank columns of token lrow in every block: 16-byte stores from where they are.  One chunk:
  // rounded to T.  Several: this chunk's fp32 partial, which a later launch on the stream (shrink_reduce_kernel, or the expand for
  // small batches) sums in index order and rounds once.
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb) {
    const int row = wrow0 + mb * 16 + lrow;
    if constexpr (NB >= 2)
      if (p.partial_through) {
        float *const part = as_global(p.partial) + ((int64_t)s * p.T + pos0 + (row & ~1)) * p.rp + kg * 4;
#pragma unroll
        for (int nb = 0; nb < NB; nb += 2)
          if (nb * 16 < p.rp) store_partials_through(part + nb * 16, p.rp, acc[mb][nb], acc[mb][nb + 1], row, cnt, lane & 1);
        continue;
      }
    if (row < cnt) {
      if (p.ksplit == 1) {
        const int t = p.out_by_token ? perm[pos0 + row] : 0;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          if (nb * 16 + kg * 4 < p.rp) store_v4<T>(p, pos0 + row, t, r, nb * 4 + kg, acc[mb][nb]);
        // columns past the tile's own rank class hold zeros, where the batch has wider ones
        for (int c4 = NB * 4 + kg; 4 * c4 < p.rp; c4 += 4) store_v4<T>(p, pos0 + row, t, r, c4, f32x4{0.f, 0.f, 0.f, 0.f});
      } else {
        float *const part = as_global(p.partial) + ((int64_t)s * p.T + pos0 + row) * p.rp + kg * 4;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          if (nb * 16 < p.rp) *reinterpret_cast<f32x4 *>(part + nb * 16) = acc[mb][nb];   // (rp: a multiple of 16)
      }
    }
  }
}

template <typename T, int NB, int MBW, bool ONCE>
__global__ __launch_bounds__(256, MBW == 2 ? 2 : 1) void shrink_gemm_kernel(const int32_t *tiles_base, int h_flags, ShrinkArgs args_in) {
  // grid (K chunks, targets, tiles).  The workgroup id mod 8 selects the XCD, so
  // with the K chunk as the fast index the tiles of an adapter that share a K chunk of A, and the
  // targets that share a K chunk of x, meet in one L2.
  const int s = (int)blockIdx.x, z_idx = (int)blockIdx.y, tile_idx = (int)blockIdx.z;
  const ShrinkArgs p = select_target(args_in, z_idx);
  __shared__ __align__(16) unsigned char lds[2 * gemm_stage_bytes(NB, MBW)];

  const int32_t *__restrict__ tile = tiles_base + (int64_t)tile_idx * TILE_WORDS;
  int r = tile[1], pos0 = tile[2], cnt = tile[3], astart = tile[4];
  if ((h_flags & SHRINK_COMPENSATE) && z_idx == 1) merged_tile(p.plan, tile_idx, 64 * MBW, r, pos0, cnt, astart);
  if (cnt <= 0) return;   // records past the last tile are zero
  // (a narrow adapter among wide ones takes the loads and products of its own rank)
  if (NB > 1 && r <= 16) shrink_gemm_tile<T, 1, MBW, ONCE>(p, s, r, pos0, cnt, astart, lds);
  else if (NB > 2 && r <= 32) shrink_gemm_tile<T, 2, MBW, ONCE>(p, s, r, pos0, cnt, astart, lds);
  else shrink_gemm_tile<T, NB, MBW, ONCE>(p, s, r, pos0, cnt, astart, lds);
}

// The same tile in eight waves, for NT targets of a call together (x is requested, written to LDS and read from it once for all
// of them), or for one of rank above 64.  Tile, K steps and order of the sums are shrink_gemm_kernel's (same bits); four pairs of
// waves split the tokens, the waves of a pair the rank columns.  One step is in flight, and a step's operands are read half by
// half, so that two workgroups share a compute unit up to 192 columns (two steps in flight at three targets of rank 64: 154
// registers, one workgroup, 5401 tokens over ranks 8-64 32.3 us against 29.3 now).
// Bound as the four-wave tile: 6.6 us of launch, look-ups, first step and partials (of one target), then the stream of x.
// 4430 tokens of rank 64, 4096 wide, four chunks, per target / together: two targets 25.8 / 23.3 us, three 33.3 / 27.5; 5401 tokens
// over ranks 8-64 25.4 / 23.6, 30.6 / 29.3.  One target of rank 128, four waves (280 registers, one workgroup a compute unit) /
// eight, the whole op: 3000 tokens over 64 adapters, 5120 wide 47.8 / 43.0; 113 shapes 0.965 in the mean.  (Up to rank 64 one target is
// better off with four waves of two 16-token blocks each: 0.98 to 1.05.)
constexpr int TARGETS_ROWS = 128;                       // tokens
constexpr int targets_half(int nt, int nb) { return (nt * nb + 1) / 2; }   // 16-column blocks of a wave
constexpr int targets_stage_bytes(int nt, int nb) { return (TARGETS_ROWS + 32 * targets_half(nt, nb)) * GEMM_KC * 2; }

// One tile and one K chunk, NB 16-row blocks of rank (of the tile's own adapter) for each of NT targets.
template <typename T, int NT, int NB, bool ONCE>
__device__ __forceinline__ void shrink_targets_tile(const ShrinkArgs &p, int s, int r, int pos0, int cnt, int astart, unsigned char *lds) {
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int KC = GEMM_KC, KS = KC / 32, C = NT * NB, HB = targets_half(NT, NB);
  constexpr int XG = 2, AG = 2 * C, APW = (AG + 7) / 8; // 8-row groups of x and A a wave loads in a step; APW waves' worth of AG
  constexpr int STAGE = targets_stage_bytes(NT, NB);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, kg = lane >> 4;           // MFMA operand roles
  const int grow = lane >> 3, gcol = lane & 7;          // loader roles: row within an 8-row group, 16-byte chunk
  const int trow0 = (wave >> 1) * 32, b0 = (wave & 1) * HB;   // products: the wave's first token row and column block
  const int32_t *__restrict__ perm = as_global(p.plan) + p.off_perm;

  const bool indexed = p.pool.a_loc_len > 0;
  const int64_t *const a_loc = indexed ? as_global(p.pool.a_loc) : reinterpret_cast<const int64_t *>(perm);
  int tok[XG], group[APW];
  int64_t prow[APW];
  bool ok[APW];
#pragma unroll
  for (int g = 0; g < XG; ++g) {
    const int row = wave * 8 * XG + g * 8 + grow;
    tok[g] = perm[pos0 + (row < cnt ? row : 0)];
  }
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    group[i] = (wave * APW + i) % AG;                   // (what goes round is loaded and written twice)
    const int z = group[i] / (2 * NB), j = group[i] % (2 * NB) * 8 + grow;
    const int slot = NT == 1 ? p.slot : z == 0 ? p.slots[0] : z == 1 ? p.slots[1] : p.slots[2];
    const int64_t idx = (int64_t)astart + (int64_t)r * slot + j;
    ok[i] = indexed && j < r && idx >= 0 && idx < p.pool.a_loc_len;
    prow[i] = a_loc[ok[i] ? idx : 0];
  }
  const uint16_t *xp[XG], *ap[APW];
  int astep[APW];                                       // all bits: the row moves on with K; none: it stays on its line
  const uint16_t *const zeros = as_global(g_zero_line) + gcol * 8;
#pragma unroll
  for (int g = 0; g < XG; ++g) xp[g] = as_global(p.x) + (uint64_t)(uint32_t)tok[g] * (uint32_t)p.h_in + gcol * 8;
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    ok[i] = ok[i] && prow[i] >= 0 && prow[i] < p.pool.w_rows;
    ap[i] = ok[i] ? as_global(p.pool.w) + (uint64_t)(uint32_t)prow[i] * (uint32_t)p.h_in + gcol * 8 : zeros;
    astep[i] = ok[i] ? -1 : 0;
  }

  const int kbeg = s * p.kchunk;
  const int kend = min(p.h_in, kbeg + p.kchunk);
  const int n_steps = (kend - kbeg) / KC;               // whole ones
  u32x4 rx[XG], ra[APW];
  auto request = [&](int step) {
    const int off = kbeg + step * KC;
#pragma unroll
    for (int g = 0; g < XG; ++g) rx[g] = ONCE ? load16_once(xp[g] + off) : load16(xp[g] + off);
#pragma unroll
    for (int i = 0; i < APW; ++i) ra[i] = load16(ap[i] + (off & astep[i]));
    requested();
  };
  // rows and chunks of a stage as in shrink_gemm_tile: x, then A block by block
  unsigned char *const wx = lds + (wave * 8 * XG + grow) * 128 + ((gcol ^ grow) << 4);
  unsigned char *wa[APW];
#pragma unroll
  for (int i = 0; i < APW; ++i) wa[i] = lds + (TARGETS_ROWS + group[i] * 8 + grow) * 128 + ((gcol ^ grow) << 4);
  const unsigned char *rxp[KS], *rap[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    rxp[ks] = lds + (trow0 + lrow) * 128 + (((ks * 4 + kg) ^ (lrow & 7)) << 4);
    rap[ks] = lds + (TARGETS_ROWS + b0 * 16 + lrow) * 128 + (((ks * 4 + kg) ^ (lrow & 7)) << 4);
  }
  f32x4 acc[2][HB];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int b = 0; b < HB; ++b) acc[mb][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto put = [&](int stage) {
#pragma unroll
    for (int g = 0; g < XG; ++g) *reinterpret_cast<u32x4 *>(wx + stage + g * 1024) = rx[g];
#pragma unroll
    for (int i = 0; i < APW; ++i) *reinterpret_cast<u32x4 *>(wa[i] + stage) = ra[i];
    requested();
  };
  auto multiply = [&](int stage) {
    // behind this barrier the stage is complete, and everybody has read the other one
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
    requested();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4 xf[2], bf[HB];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) xf[mb] = *reinterpret_cast<const u32x4 *>(rxp[ks] + stage + mb * 2048);
#pragma unroll
      for (int b = 0; b < HB; ++b) bf[b] = *reinterpret_cast<const u32x4 *>(rap[ks] + stage + b * 2048);
#pragma unroll
      for (int b = 0; b < HB; ++b)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) acc[mb][b] = Tr::mfma(as<vec8>(bf[b]), as<vec8>(xf[mb]), acc[mb][b]);
      requested();
    }
  };
  // (the loop's requests under no condition: the compiler has to know how many are outstanding where it waits)
  if (n_steps > 0) {
    int step = 0;
    request(0);
    for (; step + 1 < n_steps; ++step) {
      put((step & 1) * STAGE);
      request(step + 1);
      multiply((step & 1) * STAGE);
    }
    put((step & 1) * STAGE);
    multiply((step & 1) * STAGE);
  }
  const int off = kbeg + n_steps * KC;
  if (off < kend) {   // the end of a K that is not a multiple of 64: chunks past it read zeros
    const bool kok = off + gcol * 8 < kend;
#pragma unroll
    for (int g = 0; g < XG; ++g) rx[g] = load16(as_global(kok ? xp[g] + off : zeros));
#pragma unroll
    for (int i = 0; i < APW; ++i) ra[i] = load16(as_global(kok && astep[i] ? ap[i] + off : zeros));
    put((n_steps & 1) * STAGE);
    multiply((n_steps & 1) * STAGE);
  }
  // A lane has four consecutive rank columns of token lrow in every block: 16-byte stores from where they are.  One chunk:
  // rounded to T.  Several: this chunk's fp32 partial, which a later launch on the stream (shrink_reduce_kernel, or the expand for
  // small batches) sums in index order and rounds once.  Block b0 + b is target (b0 + b) / NB's.
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int row = trow0 + mb * 16 + lrow;
    if constexpr (NB >= 2 && HB % 2 == 0)
      if (p.partial_through) {
        float *const part = as_global(p.partial) + ((int64_t)s * p.T + pos0 + (row & ~1)) * p.rp + kg * 4;
#pragma unroll
        for (int b = 0; b < HB; b += 2) {
          const int z = (b0 + b) / NB, nb = (b0 + b) % NB;
          if (z < NT && nb * 16 < p.rp)
            store_partials_through(part + z * p.partial_tstride + nb * 16, p.rp, acc[mb][b], acc[mb][b + 1], row, cnt, lane & 1);
        }
        continue;
      }
    if (row < cnt) {
      if (NT == 1 && p.ksplit == 1) {                   // (targets go together only where K is split)
        const int t = p.out_by_token ? perm[pos0 + row] : 0;
#pragma unroll
        for (int b = 0; b < HB; ++b) {
          const int c4 = (b0 + b) * 4 + kg;
          if (b0 + b < NB && 4 * c4 < p.rp) store_v4<T>(p, pos0 + row, t, r, c4, acc[mb][b]);
        }
        // columns past the tile's own rank class hold zeros, where the batch has wider ones
        if (b0 == 0)
          for (int c4 = NB * 4 + kg; 4 * c4 < p.rp; c4 += 4) store_v4<T>(p, pos0 + row, t, r, c4, f32x4{0.f, 0.f, 0.f, 0.f});
      } else {
        float *const part = as_global(p.partial) + ((int64_t)s * p.T + pos0 + row) * p.rp + kg * 4;
#pragma unroll
        for (int b = 0; b < HB; ++b) {
          const int z = (b0 + b) / NB, nb = (b0 + b) % NB;
          if (z < NT && nb * 16 < p.rp) *reinterpret_cast<f32x4 *>(part + z * p.partial_tstride + nb * 16) = acc[mb][b];   // (rp: a multiple of 16)
        }
      }
    }
  }
}

template <typename T, int NT, int NB, bool ONCE>
__global__ __launch_bounds__(512, NT * NB <= 12 ? 4 : 2) void shrink_targets_kernel(const int32_t *tiles_base, int h_flags, ShrinkArgs args_in) {
  // grid (K chunks, groups of NT targets, tiles)
  const ShrinkArgs p = NT == 1 ? select_target(args_in, blockIdx.y) : args_in;
  __shared__ __align__(16) unsigned char lds[2 * targets_stage_bytes(NT, NB)];
  const int32_t *__restrict__ tile = tiles_base + (int64_t)blockIdx.z * TILE_WORDS;
  int r = tile[1], pos0 = tile[2], cnt = tile[3], astart = tile[4];
  const int s = (int)blockIdx.x;
  if (NT == 1 && (h_flags & SHRINK_COMPENSATE) && blockIdx.y == 1) merged_tile(p.plan, (int)blockIdx.z, TARGETS_ROWS, r, pos0, cnt, astart);
  if (cnt <= 0) return;   // records past the last tile are zero
  // (a narrow adapter among wide ones takes the loads and products of its own rank)
  if (NB > 1 && r <= 16) shrink_targets_tile<T, NT, 1, ONCE>(p, s, r, pos0, cnt, astart, lds);
  else if (NB > 2 && r <= 32) shrink_targets_tile<T, NT, 2, ONCE>(p, s, r, pos0, cnt, astart, lds);
  else if (NB > 4 && r <= 64) shrink_targets_tile<T, NT, 4, ONCE>(p, s, r, pos0, cnt, astart, lds);
  else shrink_targets_tile<T, NT, NB, ONCE>(p, s, r, pos0, cnt, astart, lds);
}

inline int head_flags(const ShrinkArgs &a) { return a.reduce_here | (a.compensate ? SHRINK_COMPENSATE : 0); }

template <typename T, int MBW>
int launch_gemm_nb(hipStream_t st, const ShrinkArgs &a, int nb, dim3 grid) {
#define MLORA_GEMM(NB)                                                                                                             \
  if (a.x_once) hipLaunchKernelGGL((shrink_gemm_kernel<T, NB, MBW, true>), grid, dim3(256), 0, st, a.plan + a.off_tiles, head_flags(a), a); \
  else hipLaunchKernelGGL((shrink_gemm_kernel<T, NB, MBW, false>), grid, dim3(256), 0, st, a.plan + a.off_tiles, head_flags(a), a)
  switch (nb) {
    case 1: MLORA_GEMM(1); break;
    case 2: MLORA_GEMM(2); break;
    case 4: MLORA_GEMM(4); break;
    default: return fail(MLORA_ERR_NO_KERNEL, "shrink: no kernel for rank blocks=%d", nb);
  }
#undef MLORA_GEMM
  return check_launch("shrink_gemm_kernel");
}

template <typename T, int MB>
int launch_shrink_nb(hipStream_t st, const ShrinkArgs &a, int nb, dim3 grid) {
  constexpr bool MAY_ONCE = MB == 1;
#define MLORA_SHRINK(MBX, NB)                                                                     \
  if (MAY_ONCE && NB > 1 && a.once_tiles <= a.n_tiles) MLORA_SHRINK_FORM(MBX, NB, (MAY_ONCE && NB > 1)); \
  else MLORA_SHRINK_FORM(MBX, NB, false)
#define MLORA_SHRINK_FORM(MBX, NB, ONCE) \
  hipLaunchKernelGGL((shrink_kernel<T, MBX, NB, ONCE>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a)
  switch (nb) {
    case 1: MLORA_SHRINK(MB, 1); break;
    case 2: MLORA_SHRINK(MB, 2); break;
    case 4: MLORA_SHRINK(MB, 4); break;
    case 8: MLORA_SHRINK((MB > 2 ? 2 : MB), 8); break;
    default: return fail(MLORA_ERR_NO_KERNEL, "shrink: no kernel for rank blocks=%d", nb);
  }
#undef MLORA_SHRINK
#undef MLORA_SHRINK_FORM
  return check_launch("shrink_kernel");
}

template <typename T, int NT>
int launch_targets(hipStream_t st, const ShrinkArgs &a, int nb, int64_t tiles) {
  const dim3 grid((unsigned)a.ksplit, (unsigned)(a.n_targets / NT), (unsigned)tiles);
#define MLORA_TARGETS(NB)                                                                                                            \
  if (a.x_once) hipLaunchKernelGGL((shrink_targets_kernel<T, NT, NB, true>), grid, dim3(512), 0, st, a.plan + a.off_tiles, head_flags(a), a); \
  else hipLaunchKernelGGL((shrink_targets_kernel<T, NT, NB, false>), grid, dim3(512), 0, st, a.plan + a.off_tiles, head_flags(a), a)
  if constexpr (NT == 1) {   // (above rank 64)
    MLORA_TARGETS(8);
  } else {
    if (nb == 1) { MLORA_TARGETS(1); }
    else if (nb == 2) { MLORA_TARGETS(2); }
    else if (nb == 4) { MLORA_TARGETS(4); }
    else { MLORA_TARGETS(8); }
  }
#undef MLORA_TARGETS
  return check_launch("shrink_targets_kernel");
}

template <typename T, int MB>
int launch_whole(hipStream_t st, const ShrinkArgs &a, int bm, int nb, int64_t tiles) {
  int shift = 0;
  while ((16 * MB) << shift < bm) ++shift;
  const int64_t pieces = tiles << shift, blocks = align_up(pieces, 8 * WHOLE_RUN);
  if (blocks > 0x7fffffff) return fail(MLORA_ERR_NO_KERNEL, "shrink: grid too large");
  const dim3 grid((unsigned)blocks);
#define MLORA_WHOLE(NB)                                                                                                        \
  hipLaunchKernelGGL((shrink_whole_kernel<T, MB, NB>), grid, dim3(64 * WHOLE_WAVES), 0, st, a.plan + a.off_tiles,             \
                     (int)pieces, shift, a)
  if (nb == 1) MLORA_WHOLE(1);
  else if constexpr (MB == 2) {
    if (nb == 2) MLORA_WHOLE(2);
    else MLORA_WHOLE(4);
  }
#undef MLORA_WHOLE
  return check_launch("shrink_whole_kernel");
}

template <typename T>
int launch_shrink_t(hipStream_t st, const ShrinkArgs &a, int bm, int nb, dim3 grid) {
  switch (bm) {
    case 16: return launch_shrink_nb<T, 1>(st, a, nb, grid);
    case 32: return launch_shrink_nb<T, 2>(st, a, nb, grid);
    case 64: return launch_shrink_nb<T, 4>(st, a, nb, grid);
    case 128: return launch_gemm_nb<T, 2>(st, a, nb, grid);
    case 256: return launch_gemm_nb<T, 4>(st, a, nb, grid);
    default: return fail(MLORA_ERR_NO_KERNEL, "shrink: tile height %d not in {16,32,64,128,256}", bm);
  }
}

}  // namespace

int launch_shrink_reduce(hipStream_t st, const ShrinkArgs &a, mlora_dtype dt) {
  if (a.T <= 0) return MLORA_OK;
  const int quarter = (int)(a.rp >> 2), rows = 256 / quarter;   // at most 32 quarters
  const dim3 grid((unsigned)((a.T + rows - 1) / rows), (unsigned)a.n_targets);
  // Partials are read as lines that nobody reads again (a pass, plain / so: 5254 tokens of rank 64 643 / 638 us, 7000 of rank 128 604 / 596,
  // 9000 of rank 64 635 / 625) where rows are whole lines (in others two workgroups share some: 2965 tokens of ranks
  // 16-48, a pass of three layers 259 us with such loads, 257 without), but not in compensations, which read few of them (a pass with / without:
  // 6368 tokens over ranks 16-64, 466 of them not the merged adapter's 751 / 746 us, 2657 1073 / 1059; 2817 of rank 128, 2 505 / 497).
  const bool once = !a.compensate && (a.rp & 31) == 0 && (reinterpret_cast<uintptr_t>(a.partial) & 127u) == 0;
#define MLORA_REDUCE_FORM(T, ONCE) \
  hipLaunchKernelGGL((shrink_reduce_kernel<T, ONCE>), grid, dim3(256), 0, st, a.plan, a.partial, quarter, 1.f / (float)quarter, head_flags(a), a.ksplit, a)
#define MLORA_REDUCE(T)                   \
  if (once) MLORA_REDUCE_FORM(T, true);   \
  else MLORA_REDUCE_FORM(T, false)
  if (dt == MLORA_F16) { MLORA_REDUCE(_Float16); }
  else { MLORA_REDUCE(__bf16); }
#undef MLORA_REDUCE_FORM
#undef MLORA_REDUCE
  return check_launch("shrink_reduce_kernel");
}

// Two or three targets of 128-token tiles together, where the fewer workgroups still fill the device evenly: two a compute unit, one
// above rank 64, so that some 270 or 540 of them need a second or third round.  How many there are depends on how many of the index's
// adapters the batch touches, which the host does not know: the least (all tokens of one adapter) must be enough, and the
// number when all adapters end in a half-empty tile not too many.  Above four K chunks a workgroup has few K steps behind its
// launch, look-ups and first loads, and sharing x gains less than the fewer workgroups lose.
// The whole op with a 256-wide output, per target / together, us.  Rank 64, three targets, 4096 wide: 140 workgroups (4400 tokens of one
// adapter) 33.2 / 36.5, 204 (4400 over 32) 43.8 / 37.9, 264 (4400 over 64) 52.8 / 57.3, 452 (14000 over 8) 77.0 / 63.7; eight chunks, 160
// (2505 over one, 8192 wide) 37.5 / 39.8; two targets 156 (4400 over 8) 35.3 / 31.1, 592 (5400 over 64, 8192 wide) 68.7 / 74.0.  Rank 128,
// three targets: 250 workgroups (14000 over 32, 8192 wide) 247 / 173, 144 (4409 over 4, 3072 wide) 41.6 / 51.6; two, eight chunks: 112
// (1276 over 7, 3072 wide) 23.0 / 27.1.  1500 shapes of 1000 to 16000 tokens, 2048 to 14336 wide, batches of one to all of up to 150 adapters,
// the ones it takes: rank up to 64 0.92 (two targets) and 0.88 (three), above 0.95 and 0.93 in the mean; 22 of 830 above 1.02, 1.10 at worst.
bool shrink_targets_together(int64_t T, int64_t adapters, int64_t max_rank, int bm, int ksplit, int n_targets) {
  if (bm != 128 || ksplit < 2 || (n_targets != 2 && n_targets != 3) || T < 64 * adapters) return false;
  const int64_t least = (T + 127) / 128 * ksplit, usual = (T / 128 + adapters / 2) * ksplit;
  const bool three = n_targets == 3, many = ksplit > 4;
  if (max_rank > 64) {
    if (usual > (many ? 240 : 256 - 2 * ksplit)) return false;   // (one round of one per unit; sizes of tails vary)
    return least >= (three ? many ? 208 : 180 : many ? 168 : 148);
  }
  if (usual > 512 && usual <= 704) return false;   // into the third round
  if (!three) return least >= 128;
  return many ? least >= 176 && (usual <= 232 || usual > 704) : least >= 160 && (usual <= 256 || usual > 336);
}

int launch_shrink(hipStream_t st, const ShrinkArgs &args, int bm, int max_rank, int64_t grid_tiles,
                  mlora_dtype dt) {
  ShrinkArgs a = args;
  a.x_once = a.partial_through = 0;
  a.once_tiles = bm == 16 ? shrink_once_tiles(a, a.n_tiles, max_rank) : 0x7fffffff;
  int nb = (max_rank + 15) / 16;
  nb = nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : 8;
  if (nb == 8 && (bm == 64 || bm == 256)) return fail(MLORA_ERR_NO_KERNEL, "shrink: rank > 64 needs tile height 16, 32 or 128");
  if (grid_tiles <= 0) return MLORA_OK;
  if (a.whole) {
    if (a.ksplit != 1 || bm < a.whole || nb > (a.whole == 64 ? 1 : 4)) return fail(MLORA_ERR_NO_KERNEL, "shrink: no whole-K kernel here");
    if (a.whole == 64) return dt == MLORA_F16 ? launch_whole<_Float16, 4>(st, a, bm, nb, grid_tiles) : launch_whole<__bf16, 4>(st, a, bm, nb, grid_tiles);
    return dt == MLORA_F16 ? launch_whole<_Float16, 2>(st, a, bm, nb, grid_tiles) : launch_whole<__bf16, 2>(st, a, bm, nb, grid_tiles);
  }
  if (a.reduce_here) grid_tiles = (grid_tiles + 7) / 8 * 8;   // ids are dealt to the 8 XCDs tile by tile
  if (grid_tiles * a.ksplit * a.n_targets > 0x7fffffff) return fail(MLORA_ERR_NO_KERNEL, "shrink: grid too large");
  dim3 grid((unsigned)(grid_tiles * a.ksplit * a.n_targets));
  if (bm >= 128) {
    if (grid_tiles > 65535) return fail(MLORA_ERR_NO_KERNEL, "shrink: grid too large");   // (4M tokens of 8192 adapters have 40960)
    grid = dim3((unsigned)a.ksplit, (unsigned)a.n_targets, (unsigned)grid_tiles);
    const bool together = !a.compensate && shrink_targets_together(a.T, grid_tiles - (a.T + 127) / 128, max_rank, bm, a.ksplit, a.n_targets);
    // x is read as lines that nobody reads again (load16_once) where that is so: not by one target's workgroups after another's, nor where
    // the caller's next call reads it (7000 tokens of rank 128 in one-call entry points 490 / 515 us a pass); in rows of whole lines; and
    // from so much of x on that the L2s do not keep it anyway.  A pass, plain / so: 5254 tokens of rank 64, seven projections of 4096 and 11008,
    // 661 / 638 us, 5401 over ranks 8-64 669 / 664, 14000, 5120 wide 1865 / 1841, 9000 of rank 64 in 256-token tiles 628 / 622; 2600 (21 MB of
    // x) 620 / 624, 1200 421 / 423.  (It is `down`, 119 MB of x, that gains, 55.6 / 40.0 us; the expands behind lose 8 us of three targets.)
    // Partials are written through in whole lines instead of left in the L2s for the end of the kernel.  A pass, plain / through: 5254 tokens
    // of rank 64 644 / 638, 7000 of rank 128 604 / 596, 1200 of rank 64 433 / 421, in one-call entry points 2600 of it 531 / 521; 3887 of rank
    // 64 whose expand sums them, once for every column chunk, 337 / 334; compensations of 6368 tokens over ranks 16-64 1081 / 1074.
    a.x_once = !a.out_by_token && (a.n_targets == 1 || together) && (int64_t)a.T * a.h_in * 2 >= L2_BYTES && !(a.h_in & 63) && !(reinterpret_cast<uintptr_t>(a.x) & 127u);
    a.partial_through = a.ksplit > 1 && (a.rp & 31) == 0 && (reinterpret_cast<uintptr_t>(a.partial) & 127u) == 0;
    if (together) {
      if (a.n_targets == 3) return dt == MLORA_F16 ? launch_targets<_Float16, 3>(st, a, nb, grid_tiles) : launch_targets<__bf16, 3>(st, a, nb, grid_tiles);
      return dt == MLORA_F16 ? launch_targets<_Float16, 2>(st, a, nb, grid_tiles) : launch_targets<__bf16, 2>(st, a, nb, grid_tiles);
    }
    if (nb == 8) return dt == MLORA_F16 ? launch_targets<_Float16, 1>(st, a, nb, grid_tiles) : launch_targets<__bf16, 1>(st, a, nb, grid_tiles);
  }
  if (a.reduce_here)
    grid = dim3((unsigned)(8 * a.ksplit), (unsigned)a.n_targets, (unsigned)(grid_tiles / 8));   // at most 4096 tokens (csrc/api.hip)
  return dt == MLORA_F16 ? launch_shrink_t<_Float16>(st, a, bm, nb, grid)
                         : launch_shrink_t<__bf16>(st, a, bm, nb, grid);
}

}  // namespace mlora
