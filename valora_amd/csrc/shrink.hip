// LoRA shrink for gfx950:  v[row, j] = T( sum_k x[t, k] * A_a[j, k] )
//
// shrink_kernel: one workgroup (4 waves) owns one adapter-grouped tile of up to 16*MB tokens and one K chunk
// (shrink_core.h has the loads and the products).  Bound by its chain of round trips, not by bytes: tile record ->
// look-ups -> operand loads -> cross-wave sum -> hand-over of the K chunks (what it measured is in shrink_core.h).
// shrink_gemm_kernel: 128- and 256-token tiles.
//
// Split-K without atomics: every workgroup writes its fp32 partial tile and is done; the chunks
// are summed in index order (bit-reproducible) by shrink_reduce_kernel or by the expand.
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

// Epilogue of the GEMM shrink.  `tile` is the workgroup's fp32 result in LDS, row-major
// with row stride ld: rows = tokens of the tile, columns = rank.
//   ksplit == 1 : rounded to T and stored.
//   ksplit  > 1 : stored as this K-chunk's fp32 partial (ordinary stores, then the workgroup is
//                 done); a later launch on the stream -- shrink_reduce_kernel, or the expand
//                 itself for small batches -- sums the chunks in index order and rounds once.
template <typename T>
__device__ __forceinline__ void shrink_epilogue(const ShrinkArgs &p, const float *tile, int ld, int s, int pos0,
                                                int cnt, int r, const int32_t *perm) {
  const int tid = threadIdx.x;
  if (p.ksplit == 1) {
    const int n_el = cnt * p.rp;
    for (int e = tid; e < n_el; e += 256) {
      const int row = e / p.rp, col = e - row * p.rp;
      store_v<T>(p, pos0 + row, p.out_by_token ? perm[pos0 + row] : 0, r, col, tile[row * ld + col]);
    }
    return;
  }
  const int quarter = p.rp >> 2;       // rp is a multiple of 16
  const int n_vec = cnt * quarter;
  f32x4 *part = reinterpret_cast<f32x4 *>(p.partial + ((int64_t)s * p.T + pos0) * p.rp);
  for (int e = tid; e < n_vec; e += 256) {
    const int row = e / quarter, c4 = e - row * quarter;
    const float *src = tile + row * ld + 4 * c4;
    part[e] = f32x4{src[0], src[1], src[2], src[3]};
  }
}

// v[row, :] = T(sum_s partial[s][row][:]) for every row that has an adapter; one thread per four columns, a workgroup the rows
// that fit whole (partial rows stand one after the other: a thread's offset in the workgroup's piece is its index).
// Bound by a launch and three round trips (arguments, chunks, store): a few MB.  Four or eight chunks are requested before any
// is used, beside the row's look-ups; no division.  With 64-bit divisions, a round trip per conditional chunk and 2-byte stores:
// 7600 tokens of rank 32 in four chunks 3.5 us a launch, now 2.7.
template <typename T>
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
      q[u] = *reinterpret_cast<const f32x4 *>(chunk + at);
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
template <typename T, int MB, int NB>
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
  shrink_tile_to_lds<T, MB, NB>(p.x, p.h_in, p.pool, p.slot, perm, r, pos0, cnt, astart, kbeg, kend, s_tile);
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

// What a rank row that is not there reads, K step after K step (one 128-byte line).
__device__ const __align__(128) uint16_t g_zero_line[64] = {};

// Prefill-sized tiles (128 tokens): GEMM structure with a three-stage LDS ring.
//
// The four waves split the tile's tokens (32 each), so no cross-wave reduction is needed.  Both
// operands of a 64-wide K step go from global memory straight into LDS with 16-byte
// global_load_lds (no registers are held while the data is in flight): every wave streams its
// own x rows into a private part of the stage, the adapter's A rows are loaded once per
// workgroup and shared by all waves.  A load instruction covers 8 rows x 128 contiguous bytes
// (whole cache lines: asking for the two halves of a line with two instructions measured up to
// 30 % slower) and writes them to LDS in lane order, so a stage holds rows of 128 bytes; the
// lane that fills 16-byte chunk c of row R fetches global chunk c ^ (R & 7), which spreads the
// later ds_read_b128 of an MFMA operand (16 rows, one chunk column) over the banks.  Two stages
// are always in flight while the third is consumed; one s_barrier per K step.
//
// Bound by what a compute unit takes in (x from HBM, A once per tile from L2: 33 GB/s measured with plain loads of this
// pattern) and, on top, by what stands between a barrier and the step's loads: masks, votes and dummy loads per
// instruction, which whole steps do without.  With that and both halves' LDS reads ahead of the products: 7600-token
// prefill over 24 adapters of rank 32 (4 layers, shrink and expand) 739 -> 712 us, 5401 tokens of mixed ranks (two
// layers, seven projections) 789 -> 760, 5254 tokens of rank 64 778 -> 766.  (Either alone: whole steps without masks
// 741 -> 716, 789 -> 766, 777 -> 769; both halves read ahead 739 -> 728, 801 -> 796, 778 -> 776.)
template <typename T, int NB, int MBW>
__global__ __launch_bounds__(256) void shrink_gemm_kernel(const int32_t *tiles_base, int h_ksplit, int h_n_targets, int h_flags, int,
                                                          ShrinkArgs args_in) {
  // workgroup id = (tile * targets + target) * ksplit + K chunk.  The id mod 8 selects the XCD, so
  // with the K chunk as the fast index the tiles of an adapter that share a K chunk of A, and the
  // targets that share a K chunk of x, meet in one L2.
  const int wg_tz = blockIdx.x / h_ksplit;
  const int tile_idx = wg_tz / h_n_targets;
  const int z_idx = wg_tz - tile_idx * h_n_targets;
  const ShrinkArgs p = select_target(args_in, z_idx);
  const int s = blockIdx.x - wg_tz * h_ksplit;
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int KC = 64, KS = KC / 32, STAGES = 3;      // MBW: 16-token blocks per wave (tile = 64 * MBW tokens)
  static_assert(KC * 2 == 128, "a K step is one 128-byte line per row");
  constexpr int XBLK = MBW * 2;                         // 8-row groups (1 KB) of x per wave per stage
  constexpr int ABLK = NB * 2;                          // 8-row groups of A per stage (shared)
  constexpr int APW = ABLK >= 4 ? ABLK / 4 : 1;         // A groups each wave loads per stage
  constexpr int A_SLOTS = APW * 4;                      // >= ABLK; surplus slots hold duplicates
  constexpr int STAGE_BYTES = (4 * XBLK + A_SLOTS) * 1024;
  constexpr int TILE_BYTES = 64 * MBW * NB * 16 * 4;
  constexpr int LOADS_PER_STAGE = XBLK + APW;           // per wave, identical for all waves
  constexpr int RING_BYTES = STAGES * STAGE_BYTES + 1024;   // + one scratch block for dummy loads
  __shared__ __align__(16) unsigned char s_raw[RING_BYTES > TILE_BYTES ? RING_BYTES : TILE_BYTES];

  const int32_t *__restrict__ tile = tiles_base + (int64_t)tile_idx * TILE_WORDS;
  int r = tile[1], pos0 = tile[2], cnt = tile[3], astart = tile[4];
  if ((h_flags & SHRINK_COMPENSATE) && z_idx == 1) merged_tile(p.plan, tile_idx, 64 * MBW, r, pos0, cnt, astart);
  if (cnt <= 0) return;   // records past the last tile are zero

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, kg = lane >> 4;           // MFMA operand roles
  const int grow = lane >> 3;                           // loader roles: row within an 8-row group,
  const int gchunk = (lane & 7) ^ grow;                 // global 16-byte chunk this lane fetches
  const int32_t *__restrict__ perm = p.plan + p.off_perm;
  const int64_t base = (int64_t)astart + (int64_t)r * p.slot;
  const int wrow0 = wave * 16 * MBW;
  const bool wave_active = wrow0 < cnt;                 // wave-uniform

  // this lane's global row pointers (already at its chunk)
  const uint16_t *xp[XBLK];
  bool xok[XBLK];
#pragma unroll
  for (int g = 0; g < XBLK; ++g) {
    const int row = wrow0 + g * 8 + grow;
    xok[g] = row < cnt;
    const int t = perm[pos0 + (xok[g] ? row : 0)];       // (a row past the tile's end reads the first one's)
    xp[g] = p.x + (int64_t)t * p.h_in + gchunk * 8;
  }
  // A groups this wave loads: slot = wave*APW + i -> rows slot*8 .. slot*8+7 of the rank
  const uint16_t *ap[APW];
  bool aok[APW];
  int astep[APW];                                       // all bits: the row moves on with K; none: it stays on its line
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    const int slot = (wave * APW + i) % ABLK;           // surplus slots duplicate real groups
    const int j = slot * 8 + grow;
    const int64_t idx = base + j;
    bool ok = j < r && idx >= 0 && idx < p.pool.a_loc_len;
    const int64_t prow = ok ? p.pool.a_loc[idx] : 0;
    ok = ok && prow >= 0 && prow < p.pool.w_rows;
    aok[i] = ok;
    // a row past the rank, or outside the index or the pool, reads zeros
    ap[i] = (ok ? p.pool.w + prow * p.h_in : g_zero_line) + gchunk * 8;
    astep[i] = ok ? -1 : 0;
  }

  const int kbeg = s * p.kchunk;
  const int kend = min(p.h_in, kbeg + p.kchunk);
  const int n_steps = (kend - kbeg + KC - 1) / KC;

  // byte offsets inside a stage: x rows of this wave, then the shared A rows
  const uint32_t ring = lds_offset(s_raw);
  const uint32_t x_off = (uint32_t)(wave * XBLK) * 1024u;
  const uint32_t a_off = (uint32_t)(4 * XBLK) * 1024u;
  const u32x4 zero4 = {0, 0, 0, 0};

  // Issue every load of one K step: EXACTLY LOADS_PER_STAGE load instructions per wave, because the
  // consumer waits with a compile-time vmcnt.  A load whose lanes are all masked off would be skipped
  // by the hardware branch around it, so in that case a dummy load into a scratch block is issued
  // instead.  Lanes beyond the end of K, and those of rank rows that are not there, write zeros into their own slot (no
  // other lane touches it).
  unsigned char *dummy = s_raw + STAGES * STAGE_BYTES;
  auto load_or_dummy = [&](bool c, const uint16_t *src, unsigned char *dst) {
    if (__builtin_amdgcn_ballot_w64(c) != 0ull) {
      if (c) __builtin_amdgcn_global_load_lds(GLOBAL_PTR(src), LDS_PTR(dst), 16, 0, 0);
    } else {
      __builtin_amdgcn_global_load_lds(GLOBAL_PTR(p.plan), LDS_PTR(dummy), 16, 0, 0);
    }
  };
  auto issue = [&](int step) {
    const int stage = step % STAGES;
    unsigned char *sbase = s_raw + stage * STAGE_BYTES;
    const int off = kbeg + step * KC;
    if (off + KC <= kend) {
      // whole steps, all but the last one of a K that is not a multiple of 64: every lane reads, x rows past the tile's end
      // the first one's (their results are never stored) and rank rows that are not there the line of zeros, so a load is
      // an address and an instruction
#pragma unroll
      for (int g = 0; g < XBLK; ++g)
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR(xp[g] + off), LDS_PTR(sbase + x_off + g * 1024), 16, 0, 0);
#pragma unroll
      for (int i = 0; i < APW; ++i)
        __builtin_amdgcn_global_load_lds(GLOBAL_PTR(ap[i] + (off & astep[i])), LDS_PTR(sbase + a_off + (wave * APW + i) * 1024), 16, 0, 0);
      return;
    }
    const int k = off + gchunk * 8;                     // first K element of this lane's chunk
    const bool kok = k < kend;
#pragma unroll
    for (int g = 0; g < XBLK; ++g) {
      unsigned char *dst = sbase + x_off + g * 1024;
      load_or_dummy(xok[g] && kok, xp[g] + kbeg + step * KC, dst);
      if (!kok) lds_write16(lds_offset(dst) + lane * 16, zero4);
    }
#pragma unroll
    for (int i = 0; i < APW; ++i) {
      unsigned char *dst = sbase + a_off + (wave * APW + i) * 1024;
      load_or_dummy(aok[i] && kok, ap[i] + kbeg + step * KC, dst);
      if (!(aok[i] && kok)) lds_write16(lds_offset(dst) + lane * 16, zero4);
    }
  };
  // where the MFMA operand (row R of a region, K block ks) of this lane sits inside a stage
  auto frag_off = [&](int R, int ks) -> uint32_t {
    return (uint32_t)R * 128u + (uint32_t)(((ks * 4 + kg) ^ (R & 7)) * 16);
  };

  f32x4 acc[MBW][NB];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  issue(0);
  if (n_steps > 1) issue(1);
  for (int step = 0; step < n_steps; ++step) {
    // wait for this step's loads (the next step's may stay in flight), then meet the other waves:
    // after the barrier the stage is complete for everybody and the stage consumed in the previous
    // iteration is free to be refilled
    if (step + 1 < n_steps) wait_vmcnt<LOADS_PER_STAGE>(); else wait_vmcnt<0>();
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
    if (step + 2 < n_steps) issue(step + 2);
    const int stage = step % STAGES;
    if (wave_active) {
      // both halves' operands are requested before the first half is used
      u32x4 xfs[KS][MBW], bfs[KS][NB];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb)
          xfs[ks][mb] = lds_read16(ring + stage * STAGE_BYTES + x_off + frag_off(mb * 16 + lrow, ks));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          bfs[ks][nb] = lds_read16(ring + stage * STAGE_BYTES + a_off + frag_off(nb * 16 + lrow, ks));
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) wait_lgkmcnt<MBW + NB>(); else wait_lgkmcnt<0>();
        u32x4 (&xf)[MBW] = xfs[ks];
        u32x4 (&bf)[NB] = bfs[ks];
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb) pin(xf[mb]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) pin(bf[nb]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          if (nb * 16 < r) {
#pragma unroll
            for (int mb = 0; mb < MBW; ++mb)
              acc[mb][nb] = Tr::mfma(as<vec8>(xf[mb]), as<vec8>(bf[nb]), acc[mb][nb]);
          }
        }
      }
    }
  }
  wait_lgkmcnt0();
  __syncthreads();   // everybody is done reading the ring: reuse it for the result tile

  float *otile = reinterpret_cast<float *>(s_raw);
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = wrow0 + mb * 16 + kg * 4 + i;
        const int col = nb * 16 + lrow;
        otile[row * (NB * 16) + col] = acc[mb][nb][i];
      }
  __syncthreads();
  shrink_epilogue<T>(p, otile, NB * 16, s, pos0, cnt, r, perm);
}

inline int head_flags(const ShrinkArgs &a) { return a.reduce_here | (a.compensate ? SHRINK_COMPENSATE : 0); }

template <typename T, int MBW>
int launch_gemm_nb(hipStream_t st, const ShrinkArgs &a, int nb, dim3 grid) {
  switch (nb) {
    case 1: hipLaunchKernelGGL((shrink_gemm_kernel<T, 1, MBW>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    case 2: hipLaunchKernelGGL((shrink_gemm_kernel<T, 2, MBW>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    case 4: hipLaunchKernelGGL((shrink_gemm_kernel<T, 4, MBW>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    case 8:
      if constexpr (MBW <= 2) {
        hipLaunchKernelGGL((shrink_gemm_kernel<T, 8, MBW>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a);
        break;
      }
      return fail(MLORA_ERR_NO_KERNEL, "shrink: rank > 64 has no 256-token tile");
    default: return fail(MLORA_ERR_NO_KERNEL, "shrink: no kernel for rank blocks=%d", nb);
  }
  return check_launch("shrink_gemm_kernel");
}

template <typename T, int MB>
int launch_shrink_nb(hipStream_t st, const ShrinkArgs &a, int nb, dim3 grid) {
  switch (nb) {
    case 1: hipLaunchKernelGGL((shrink_kernel<T, MB, 1>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    case 2: hipLaunchKernelGGL((shrink_kernel<T, MB, 2>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    case 4: hipLaunchKernelGGL((shrink_kernel<T, MB, 4>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    case 8: hipLaunchKernelGGL((shrink_kernel<T, (MB > 2 ? 2 : MB), 8>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.ksplit, a.n_targets, head_flags(a), a.n_tiles, a); break;
    default: return fail(MLORA_ERR_NO_KERNEL, "shrink: no kernel for rank blocks=%d", nb);
  }
  return check_launch("shrink_kernel");
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
#define MLORA_REDUCE(T) \
  hipLaunchKernelGGL(shrink_reduce_kernel<T>, grid, dim3(256), 0, st, a.plan, a.partial, quarter, 1.f / (float)quarter, head_flags(a), a.ksplit, a)
  if (dt == MLORA_F16) MLORA_REDUCE(_Float16);
  else MLORA_REDUCE(__bf16);
#undef MLORA_REDUCE
  return check_launch("shrink_reduce_kernel");
}

int launch_shrink(hipStream_t st, const ShrinkArgs &a, int bm, int max_rank, int64_t grid_tiles,
                  mlora_dtype dt) {
  int nb = (max_rank + 15) / 16;
  nb = nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : 8;
  if (nb == 8 && (bm == 64 || bm == 256)) return fail(MLORA_ERR_NO_KERNEL, "shrink: rank > 64 needs tile height 16, 32 or 128");
  if (grid_tiles <= 0) return MLORA_OK;
  if (a.reduce_here) grid_tiles = (grid_tiles + 7) / 8 * 8;   // ids are dealt to the 8 XCDs tile by tile
  if (grid_tiles * a.ksplit * a.n_targets > 0x7fffffff) return fail(MLORA_ERR_NO_KERNEL, "shrink: grid too large");
  dim3 grid((unsigned)(grid_tiles * a.ksplit * a.n_targets));
  if (a.reduce_here)
    grid = dim3((unsigned)(8 * a.ksplit), (unsigned)a.n_targets, (unsigned)(grid_tiles / 8));   // at most 4096 tokens (csrc/api.hip)
  return dt == MLORA_F16 ? launch_shrink_t<_Float16>(st, a, bm, nb, grid)
                         : launch_shrink_t<__bf16>(st, a, bm, nb, grid);
}

}  // namespace mlora
