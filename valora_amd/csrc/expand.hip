// LoRA expand for gfx950:  y[t, o] = T( y[t, o] + scale_a * sum_{j<r} T(v[t, j]) * B_a[j, o] )
//
// The pool stores a slot's B block as [H_out, r] row-major spread over r pool rows, so output
// column o owns r consecutive elements at flat offset o*r: the B operand of the MFMA (column =
// output, 8 consecutive rank elements per lane) is again one 16-byte global load per lane, and
// 16 neighbouring outputs are one contiguous 32*r-byte run.  A workgroup owns one adapter-grouped
// tile of tokens and 256 output columns (64 per wave); each wave loads its B fragments once into
// registers and reuses them for every 16-token block of the tile.  The fp32 MFMA result is
// turned through a small LDS tile so that the read-modify-write of y is done with 16-byte
// accesses of 128 contiguous bytes per token row; the add is done in fp32 and rounded once.
//
// v is a T matrix: either the shrink's internal buffer (rows in sorted-position order; rounded
// to T once, as the reference does by holding `delta` in a T tensor between its two launches)
// or a matrix supplied by the caller (rows in token order).
//
// Reference semantics: valora/csrc/bgmv/bgmv_impl.cuh:152-207.
#include "expand_core.h"
#include "kernel_common.h"

namespace mlora {

namespace {

constexpr int EXP_BN = 256;       // outputs per workgroup
constexpr int EXP_WN = 64;        // outputs per wave
constexpr int STAGE_LD = EXP_WN + 4;
constexpr int EXP_MBU = 2;         // 16-token blocks whose loads are in flight together
constexpr int EXP_MAX_BM = 256;   // tallest expand tile (tokens), one thread per token at set-up


// the arguments of target z of a multi-target launch
__device__ __forceinline__ ExpandArgs select_target(const ExpandArgs &a, int z) {
  ExpandArgs p = a;
  p.slot = a.slots[z];
  p.y = a.ys[z];
  p.pool.w = a.ws[z];
  p.pool.w_rows = a.w_rows_t[z];
  p.v = a.v + (int64_t)z * a.v_tstride;
  if (a.partial) p.partial = a.partial + (int64_t)z * a.partial_tstride;
  return p;
}

// Waves per SIMD the register allocator has to leave room for.  The rank-64 variant that reads a finished
// v sits 2 registers above the 96 that allow 5 waves; held to 5 it measured 1-6 % faster on the prefill and
// mixed shapes (more workgroups resident per round), at 6 it spills.  The rank-32 one fits 7 (at 5 a 6749-token prefill
// takes 27.5 instead of 26 us), and the one that sums partials 4.
constexpr int expand_min_waves(int kb, bool partial, bool comp) {
  return comp ? 1 : kb == 2 && !partial ? 5 : kb == 1 ? (partial ? 4 : 7) : 1;
}

// COMP: the compensation of a request whose base weights hold another adapter (csrc/api.hip, mlora_lora_compensate):
// y = T(T(y + own scale * v B_own) - merged scale * v' B_merged), where v' is the "target" 1 matrix of the same positions:
// both products in one pass over y.
template <typename T, int KB, bool PARTIAL, bool COMP>
__global__ __launch_bounds__(256, expand_min_waves(KB, PARTIAL, COMP)) void expand_kernel(const int32_t *tiles_base, int h_n_ochunks,
                                                                                    ExpandArgs args_in) {
  // (tiles_base, h_n_ochunks: what the first dependent load needs, in front so that kernel-argument preloading
  // delivers them in registers)
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  __shared__ float stage[4][16][STAGE_LD];
  __shared__ int32_t s_perm[EXP_MAX_BM];

  const int tile_idx = blockIdx.x / h_n_ochunks;
  const int oc = blockIdx.x - tile_idx * h_n_ochunks;
  const int32_t *__restrict__ tile = tiles_base + (int64_t)tile_idx * TILE_WORDS;
  const int a = tile[0], r = tile[1], pos0 = tile[2], astart = tile[4];
  const int cnt = COMP ? abs(tile[3]) : tile[3];   // (negative: no usable rank of its own, r = 0)
  if (cnt <= 0) return;   // records past the last tile are zero
  const ExpandArgs p = select_target(args_in, blockIdx.y);
  constexpr int MBU = COMP && KB == 4 ? 1 : EXP_MBU;   // two rank-128 operand sets leave registers for one block
  const int rk = min(r, p.kmax);  // rank columns the narrow operand really has (bgmv_impl.cuh:167,186)

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, kg = lane >> 4;
  const int64_t base = (int64_t)astart + (int64_t)r * p.slot;
  const int o_wave = oc * EXP_BN + wave * EXP_WN;

  // Everything that depends only on the tile header is requested first, in one round trip:
  // the tile's token indices, the pool rows of the B fragments and the scale.
  int my_perm = 0;
  if (tid < cnt) my_perm = p.plan[p.off_perm + pos0 + tid];
  const float scale = Tr::to_float(p.scales[a]);
  const float inv_h_out = 1.0f / (float)p.h_out;
  int64_t brow[4][KB];
  uint32_t boff[4][KB];
  auto look_up = [&](int rr, int rrk, int64_t rbase, int64_t (&row)[4][KB], uint32_t (&off)[4][KB]) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const int o = o_wave + nb * 16 + lrow;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int j0 = kb * 32 + kg * 8;
        row[nb][kb] = -1;
        off[nb][kb] = 0;
        if (o < p.h_out && j0 < rrk) {
          const uint32_t flat = (uint32_t)o * (uint32_t)rr + (uint32_t)j0;   // < 2^16 * 2^7
          uint32_t bin;
          divmod24(flat, (uint32_t)p.h_out, inv_h_out, bin, off[nb][kb]);
          const int64_t idx = rbase + bin;
          if (idx >= 0 && idx < p.pool.a_loc_len) row[nb][kb] = p.pool.a_loc[idx];
        }
      }
    }
  };
  look_up(r, rk, base, brow, boff);
  int64_t brow2[COMP ? 4 : 1][COMP ? KB : 1];
  uint32_t boff2[COMP ? 4 : 1][COMP ? KB : 1];
  int rk2 = 0;
  float scale2 = 0.f;
  if constexpr (COMP) {
    const int r2 = p.plan[H_MERGED_RANK];
    rk2 = min(r2, p.kmax);
    if (r2 > 0) scale2 = -Tr::to_float(p.scales[p.plan[H_MERGED]]);
    look_up(r2, rk2, (int64_t)p.plan[H_MERGED_START] + (int64_t)r2 * p.slot, brow2, boff2);
  }
  s_perm[tid] = my_perm;
  // The only workgroup-wide barrier: it also drains the loads above (which everything below needs
  // anyway).  No barrier may follow the bulk loads below -- a barrier waits for all outstanding
  // global loads and would serialise the B, y and v traffic into separate round trips.
  __syncthreads();

  // B fragments: bfrag[nb][kb] = B^T[o = o_wave + nb*16 + lrow][j0 .. j0+8), j0 = kb*32 + kg*8
  u32x4 bfrag[4][KB], bfrag2[COMP ? 4 : 1][COMP ? KB : 1];
  auto load_b = [&](const int64_t (&brw)[4][KB], const uint32_t (&off)[4][KB], u32x4 (&frag)[4][KB]) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int64_t row = brw[nb][kb];
        frag[nb][kb] = (row >= 0 && row < p.pool.w_rows) ? load16(p.pool.w + row * p.h_out + off[nb][kb])
                                                          : u32x4{0, 0, 0, 0};
      }
  };
  load_b(brow, boff, bfrag);
  if constexpr (COMP) load_b(brow2, boff2, bfrag2);

  // row-major roles for the y read-modify-write: 8 lanes x 16 B cover one token row of the wave's
  // 64 outputs; a wave covers 8 rows per access, two accesses per 16-token block.
  const int rr0 = lane >> 3, c8 = (lane & 7) * 8;
  const bool ocol_ok = (o_wave + c8) < p.h_out;

  // Two 16-token blocks per iteration: their y rows and v fragments are all requested before either
  // block is consumed, so an iteration costs one memory round trip for 32 tokens.
  const int n_mb = (cnt + 15) >> 4;
  for (int mb0 = 0; mb0 < n_mb; mb0 += MBU) {
    u32x4 yv[MBU][2];
    uint16_t *yp[MBU][2];
    bool yok[MBU][2];
    u32x4 vfrag[MBU][KB], vfrag2[COMP ? MBU : 1][COMP ? KB : 1];
#pragma unroll
    for (int b = 0; b < MBU; ++b) {
      const int mb = mb0 + b;
      // ---- y rows first (the longest-latency loads of the iteration)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = mb * 16 + rr0 + 8 * h;
        yok[b][h] = ocol_ok && row < cnt;
        const int t = yok[b][h] ? s_perm[row] : 0;
        yp[b][h] = p.y + (int64_t)t * p.h_out + o_wave + c8;
        yv[b][h] = yok[b][h] ? load16(yp[b][h]) : u32x4{0, 0, 0, 0};
      }
      // ---- v fragments: rows = tokens (lrow), 8 consecutive rank elements per lane
      const int prow = mb * 16 + lrow;
      const bool pok = prow < cnt;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int j0 = kb * 32 + kg * 8;
        u32x4 v = {0, 0, 0, 0};
        if (pok && j0 < rk) {
          if constexpr (PARTIAL) {
            // split-K partials of the shrink: all chunks are requested before any is consumed,
            // summed in chunk order and rounded to T once
            float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            const float *src0 = p.partial + ((int64_t)pos0 + prow) * p.rp + j0;
            const int64_t sstride = (int64_t)p.T * p.rp;
            for (int s0 = 0; s0 < p.ksplit; s0 += 4) {
              f32x4 lo[4], hi[4];
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const bool ok = s0 + u < p.ksplit;
                const f32x4 *src = reinterpret_cast<const f32x4 *>(src0 + (int64_t)(s0 + u) * sstride);
                lo[u] = ok ? src[0] : f32x4{0.f, 0.f, 0.f, 0.f};
                hi[u] = ok ? src[1] : f32x4{0.f, 0.f, 0.f, 0.f};
              }
#pragma unroll
              for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) { f[i] += lo[u][i]; f[4 + i] += hi[u][i]; }
            }
            v = pack8<T>(f);
          } else {
            const int64_t vrow = p.v_by_pos ? (int64_t)(pos0 + prow) : (int64_t)s_perm[prow];
            v = load16(p.v + vrow * p.v_stride + j0);
          }
        }
        vfrag[b][kb] = v;
        if constexpr (COMP)   // the same positions' rows of the merged adapter's matrix
          vfrag2[b][kb] = (pok && j0 < rk2) ? load16(p.v + p.v_tstride + (int64_t)(pos0 + prow) * p.v_stride + j0)
                                            : u32x4{0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int b = 0; b < MBU; ++b) {
      if (mb0 + b < n_mb) {   // workgroup-uniform
        // ---- delta block through the matrix cores, turned through LDS into token-major order and added to the y rows
        auto add = [&](const u32x4 (&vf)[KB], const u32x4 (&bf)[4][KB], int rkk, float sc, bool last) {
#pragma unroll
          for (int nb = 0; nb < 4; ++nb) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
              if (kb * 32 < rkk) acc = Tr::mfma(as<vec8>(vf[kb]), as<vec8>(bf[nb][kb]), acc);
#pragma unroll
            for (int i = 0; i < 4; ++i) stage[wave][kg * 4 + i][nb * 16 + lrow] = acc[i];
          }
          // stage[wave] is private to this wave and a wave's LDS operations execute in order, so only
          // the compiler has to be kept from reordering the reads below over the writes above.
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (yok[b][h]) {
              const float *srow = &stage[wave][rr0 + 8 * h][c8];
              float f[8];
              unpack8<T>(yv[b][h], f);
#pragma unroll
              for (int i = 0; i < 8; ++i) f[i] += sc * srow[i];
              if (last) store16(yp[b][h], pack8<T>(f));
              else yv[b][h] = pack8<T>(f);
            }
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
        };
        if (!COMP || rk > 0) add(vfrag[b], bfrag, rk, scale, !COMP);
        if constexpr (COMP) add(vfrag2[b], bfrag2, rk2, scale2, true);
      }
    }
  }
}

// Tiles of 16 tokens (decode batches).  Four independent waves of 64 outputs each: no LDS, no barrier (expand_core.h has
// the loads and the product, and what it measured).  Grid: (column chunks, tiles, targets).
// (Two or four column chunks a workgroup, all their loads in flight together, lose wherever the narrow operand is finished: 512
// tokens, q+k+v at rank 16 26.1 / 27.5 us with its shrink, one target of 256 tokens, 11008 columns 8.6 / 9.6, ranks 8-64, gate+up
// of 13824 columns 25.2 / 27.4.)
constexpr int64_t SMALL_MAX_TILES = 65535;   // tiles of one launch: grid y is 16 bits
constexpr int small_min_waves(int kb, bool wide, bool comp) {   // as many as do without spills
  return comp ? (kb <= 1 ? 7 : 1) : kb <= 1 ? 8 : kb == 2 ? (wide ? 6 : 5) : (wide ? 4 : 3);
}
template <typename T, int KB, bool WIDE, bool PARTIAL, bool COMP>
__global__ __launch_bounds__(256, small_min_waves(KB, WIDE, COMP)) void expand_small_kernel(const int32_t *tiles_base, const int32_t *perm,
                                                                                         const int64_t *a_loc, int h_n_loc, int h_out,
                                                                                         ExpandArgs p) {
  using Tr = Traits<T>;
  constexpr int FKB = SmallB<KB>::FRAG_KB;
  const int tile_idx = (int)blockIdx.y, z = (int)blockIdx.z;
  // One scalar round trip: the tile record and every argument the wave is going to use (csrc/decode.hip has the reason for the asm).
  const int32_t *__restrict__ tile = tiles_base + (int64_t)tile_idx * TILE_WORDS;
  int ad = tile[0], r = tile[1], pos0 = tile[2], cnt = tile[3], astart = tile[4];
  int slot = p.slots[z], kmax = p.kmax, w_rows = (int)p.w_rows_t[z], v_by_pos = p.v_by_pos;
  uint16_t *y = p.ys[z];
  const uint16_t *w = p.ws[z], *v = p.v, *scales = p.scales;
  int64_t v_tstride = p.v_tstride, v_stride = p.v_stride;
  float inv_h_out = p.inv_h_out;
  asm volatile("" : "+s"(ad), "+s"(r), "+s"(pos0), "+s"(cnt), "+s"(astart), "+s"(slot), "+s"(kmax), "+s"(w_rows), "+s"(v_by_pos),
                    "+s"(y), "+s"(w), "+s"(v), "+s"(scales), "+s"(v_tstride), "+s"(v_stride), "+s"(inv_h_out));
  if (COMP) cnt = abs(cnt);                  // (negative: no usable rank of its own, r = 0)
  if (cnt <= 0) return;                      // records past the last tile are zero
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int m = lane & 15, kg = lane >> 4;
  const uint32_t o_wave = blockIdx.x * (uint32_t)EXP_BN + (uint32_t)(wave * EXP_WN);
  if (o_wave >= (uint32_t)h_out) return;
  y = as_global(y);
  w = as_global(w);
  v = as_global(v);
  scales = as_global(scales);
  const bool on = m < cnt;                   // lanes without a token work on the tile's first one and store nothing
  const int tok = perm[pos0 + (on ? m : 0)];
  const float scale = Tr::to_float(scales[ad]);
  const SmallPool pool = {w, a_loc, (uint32_t)h_n_loc, (uint32_t)w_rows, (uint32_t)h_out, inv_h_out, (uint32_t)(astart + r * slot), r,
                          min(r, kmax)};
  SmallRows<KB, WIDE> rows, rows2;
  small_look_up<KB, WIDE>(pool, o_wave, lane, rows);
  // COMP: y = T(T(y + own scale * v B_own) - merged scale * v' B_merged), as in expand_kernel
  SmallPool pool2 = pool;
  float scale2 = 0.f;
  if constexpr (COMP) {
    const int r2 = p.plan[H_MERGED_RANK];
    pool2.r = r2;
    pool2.rk = min(r2, kmax);
    pool2.base = (uint32_t)(p.plan[H_MERGED_START] + r2 * slot);
    if (r2 > 0) scale2 = -Tr::to_float(scales[p.plan[H_MERGED]]);
    small_look_up<KB, WIDE>(pool2, o_wave, lane, rows2);
  }
  const uint32_t pos = (uint32_t)(pos0 + (on ? m : 0)), vrow = v_by_pos ? pos : (uint32_t)tok;
  auto load_v = [&](const uint16_t *src, int rk, u32x4 (&f)[FKB]) {
#pragma unroll
    for (int kb = 0; kb < FKB; ++kb) {
      const int j0 = kb * 32 + kg * 8;
      f[kb] = load16(small_source(j0 < rk, src + (uint64_t)vrow * (uint64_t)v_stride + j0));
    }
  };
  u32x4 vfrag[FKB];
  if constexpr (PARTIAL)
    small_v_partials<T, KB>(as_global(p.partial) + z * p.partial_tstride + (int64_t)pos0 * p.rp, (uint32_t)((on ? m : 0) * p.rp),
                            (int64_t)p.T * p.rp, p.ksplit, pool.rk, lane, vfrag);
  else
    load_v(v + z * v_tstride, pool.rk, vfrag);
  SmallY<KB> yy;
  small_load_y(yy, y, tok, on, o_wave, (uint32_t)h_out, lane);
  requested();
  u32x4 raw[SmallB<KB>::LOADS];
  small_load_b<KB, WIDE>(pool, lane, rows, raw);
  f32x4 acc[4];
  if constexpr (COMP) {
    u32x4 vfrag2[FKB], raw2[SmallB<KB>::LOADS];
    load_v(v + v_tstride, pool2.rk, vfrag2);
    small_load_b<KB, WIDE>(pool2, lane, rows2, raw2);
    requested();
    if (pool.rk > 0) {
      small_product<T, KB>(raw, vfrag, pool.rk, lane, acc);
      small_add<T, KB>(yy, acc, scale);
    }
    small_product<T, KB>(raw2, vfrag2, pool2.rk, lane, acc);
    small_add<T, KB>(yy, acc, scale2);
  } else {
    requested();
    small_product<T, KB>(raw, vfrag, pool.rk, lane, acc);
    small_add<T, KB>(yy, acc, scale);
  }
  small_store_y(yy);
}

template <typename T, int KB>
int launch_small_kb(hipStream_t st, const ExpandArgs &a, int64_t tiles) {
  // an index without entries: the kernel reads one all the same, and drops it
  const int64_t *a_loc = a.pool.a_loc_len > 0 ? a.pool.a_loc : reinterpret_cast<const int64_t *>(a.plan + a.off_perm);
#define MLORA_SMALL(WIDE, PARTIAL, COMP)                                                                        \
  hipLaunchKernelGGL((expand_small_kernel<T, KB, WIDE, PARTIAL, COMP>), grid, dim3(256), 0, st, records,        \
                     a.plan + a.off_perm, a_loc, (int)a.pool.a_loc_len, a.h_out, a)
#define MLORA_SMALL_WIDTH(PARTIAL, COMP)                             \
  if (KB > 0 && a.h_out >= SMALL_WIDE) MLORA_SMALL((KB > 0), PARTIAL, COMP); \
  else MLORA_SMALL(false, PARTIAL, COMP)
  // Exactly as many workgroups as there are records: what stands behind the last one is no record (the words of the one-launch
  // op do, and a call of that kind leaves them non-zero).  More tiles than a grid's y takes (a million tokens) are several launches.
  for (int64_t t0 = 0; t0 < tiles; t0 += SMALL_MAX_TILES) {
    const int32_t *records = a.plan + a.off_tiles + t0 * TILE_WORDS;
    const dim3 grid((unsigned)a.n_ochunks, (unsigned)(tiles - t0 < SMALL_MAX_TILES ? tiles - t0 : SMALL_MAX_TILES), (unsigned)a.n_targets);
    if (a.compensate) { MLORA_SMALL_WIDTH(false, true); }
    else if (a.partial) { MLORA_SMALL_WIDTH(true, false); }
    else { MLORA_SMALL_WIDTH(false, false); }
  }
#undef MLORA_SMALL_WIDTH
#undef MLORA_SMALL
  return check_launch("expand_small_kernel");
}

template <typename T>
int launch_small_t(hipStream_t st, const ExpandArgs &a, int max_rank, int64_t tiles) {
  if (max_rank <= 16) return launch_small_kb<T, 0>(st, a, tiles);
  if (max_rank <= 32) return launch_small_kb<T, 1>(st, a, tiles);
  if (max_rank <= 64) return launch_small_kb<T, 2>(st, a, tiles);
  return launch_small_kb<T, 4>(st, a, tiles);
}

template <typename T>
int launch_expand_t(hipStream_t st, const ExpandArgs &a, int kb, dim3 grid) {
#define MLORA_EXPAND(KB, PARTIAL, COMP)                                                                              \
  hipLaunchKernelGGL((expand_kernel<T, KB, PARTIAL, COMP>), grid, dim3(256), 0, st, a.plan + a.off_tiles, a.n_ochunks, a)
#define MLORA_EXPAND_KB(KB)                                                                                          \
  if (a.compensate) MLORA_EXPAND(KB, false, true);                                                                   \
  else if (a.partial) MLORA_EXPAND(KB, true, false);                                                                 \
  else MLORA_EXPAND(KB, false, false)
  switch (kb) {
    case 1: MLORA_EXPAND_KB(1); break;
    case 2: MLORA_EXPAND_KB(2); break;
    case 4: MLORA_EXPAND_KB(4); break;
    default: return fail(MLORA_ERR_NO_KERNEL, "expand: no kernel for %d rank blocks", kb);
  }
#undef MLORA_EXPAND_KB
#undef MLORA_EXPAND
  return check_launch("expand_kernel");
}

}  // namespace

int launch_expand(hipStream_t st, const ExpandArgs &a, int max_rank, int64_t grid_tiles, int bm_expand, mlora_dtype dt) {
  int kb = (max_rank + 31) / 32;
  kb = kb <= 1 ? 1 : kb <= 2 ? 2 : 4;
  if (grid_tiles <= 0) return MLORA_OK;
  if (bm_expand == 16)
    return dt == MLORA_F16 ? launch_small_t<_Float16>(st, a, max_rank, grid_tiles) : launch_small_t<__bf16>(st, a, max_rank, grid_tiles);
  const int64_t blocks = grid_tiles * a.n_ochunks;
  if (blocks > 0x7fffffff) return fail(MLORA_ERR_NO_KERNEL, "expand: grid too large");
  dim3 grid((unsigned)blocks, (unsigned)a.n_targets);
  return dt == MLORA_F16 ? launch_expand_t<_Float16>(st, a, kb, grid)
                         : launch_expand_t<__bf16>(st, a, kb, grid);
}

int expand_bn() { return EXP_BN; }

}  // namespace mlora
