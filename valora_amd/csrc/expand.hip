// LoRA expand for gfx950:  y[t, o] = T( y[t, o] + scale_a * sum_{j<r} T(v[t, j]) * B_a[j, o] )
//
// The pool stores a slot's B block as [H_out, r] row-major spread over r pool rows, so output
// column o owns r consecutive elements at flat offset o*r: a B operand of the MFMA (row =
// output, 8 consecutive rank elements per lane) is again one 16-byte global load per lane.
// A workgroup owns one adapter-grouped
// tile of tokens and 256 output columns (64 per wave); each wave loads its B fragments once into
// registers and reuses them for every 16-token block of the tile; the tile's v rows are loaded once
// per workgroup into LDS.  The fp32 MFMA result is
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
constexpr int64_t MAX_GRID_TILES = 65535;   // tiles of one launch: grid y is 16 bits
constexpr int EXP_V_BATCH = 3;     // chunks of v a thread requests together
__host__ __device__ constexpr int expand_v_chunks(int kb) { return kb * 4 + 1; }   // LDS chunks of a v row, odd

// Waves per SIMD the register allocator has to leave room for: as many as do without spills of vector registers.  (Rank above 64
// with outputs narrower than SMALL_WIDE: 16 look-ups' masks do not fit the scalar registers either, 27 scalars with partial sums and 58
// with COMP stand in lanes of vector registers.  250 calls of such ranks with 256 to 1536 outputs take 0.83 of the time of masked loads.)
constexpr int expand_min_waves(int kb, bool partial, bool comp) {
  return comp || partial ? 1 : kb == 1 ? 6 : kb == 2 ? 5 : 1;
}

// Tall tiles.  One scalar round trip (record, arguments), one of look-ups and v, one for B and the first y rows; then a loop
// over 32 tokens.
// Bound by the y stream (43 MB in place take 18.1 us as one linear pass, 231 MB 81), and before that by its own instructions and by v:
// with a masked load for every unit, a look-up per unit and v as MFMA operands by every wave it had 670 instructions in front of
// the loop and 450 per 32 tokens; now 500 and 190.  Cold layers, before / now, us a launch: 6749 tokens of rank 32, 4096 columns, 32-token
// tiles 26.3 / 25.1; 5254 tokens of rank 64, 96-token tiles, one target of 4096 columns 26.4 / 22.7, three 67.4 / 57.3, two of 11008
// 108.8 / 99.4; 5401 tokens over ranks 8-64 24.8 / 22.6, 57.9 / 54.5, 93.0 / 90.9; 10000 tokens over 8 adapters of rank 128, shrink and
// expand 106 / 92.  (Of the 109 us, B and v together were 29, v alone 8.  One more or one less waves' worth of registers spills or gains
// nothing; 16 instead of 8 staged tokens, 8.7 KB more LDS, 1 % slower.)
// THROUGH: y is written through (write_through, expand_core.h) instead of left dirty in the L2s for the end of the kernel.  A pass, plain /
// through (with ONCE where it is on): 5401 tokens over ranks 8-64, seven projections of 4096 and 11008, 686 / 664 us; 5254 of rank 64 660 / 638;
// 14000 over ranks 8-64, 5120 wide 1878 / 1840; 3887 of rank 64 whose chunks are summed here (PARTIAL) 340 / 334; 1200 of rank 64 433 / 421.
// What it gives stands mostly in the next launch: of the first batch three targets of 4096 columns take 60.9 / 57.5 us, two of 11008
// 97.1 / 93.1, one 24.5 / 22.1, but 49.6, 87.7 and 20.8 where the shrinks read x the plain way, which lose more than that (csrc/shrink.hip).
// ONCE: and y is read as lines that nobody reads again (load16_once), so that the caches keep B and v, from L2_BYTES on, since less
// of it stays there until it is written; not where the chunks are summed here (0.996).  A pass, plain reads / these: 5401 tokens over
// ranks 8-64 676 / 664 us, 14000 1870 / 1840, 7000 of rank 128 604 / 596; with less of y in a launch they lose: 1200 tokens of rank 64, 3072
// wide, in calls of one target 395 / 406, 2600 520 / 530.  (Forms of their own: above rank 64 no scalar register is left for a flag.  In
// 16-token tiles such reads are 0.995.)
// COMP: the compensation of a request whose base weights hold another adapter (csrc/api.hip, mlora_lora_compensate):
// y = T(T(y + own scale * v B_own) - merged scale * v' B_merged), where v' is the "target" 1 matrix of the same positions:
// both products in one pass over y.
template <typename T, int KB, bool WIDE, bool PARTIAL, bool COMP, bool THROUGH, bool ONCE>
__global__ __launch_bounds__(256, expand_min_waves(KB, PARTIAL, COMP)) void expand_kernel(const int32_t *tiles_base, const int32_t *perm,
                                                                                    const int64_t *a_loc, int h_n_loc, int h_out,
                                                                                    ExpandArgs p) {
  // (the leading parameters: what the first dependent loads need; kernel-argument preloading delivers them in registers)
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int MBU = COMP && KB == 4 ? 1 : EXP_MBU;   // two rank-128 operand sets leave registers for one block
  constexpr int VC = KB * 4, VLD = expand_v_chunks(KB);
  __shared__ __align__(16) float stage[4][8][STAGE_LD];
  // The tile's v rows, with COMP the merged adapter's behind them, and its token indices.  (96 tokens of rank 64
  // are 22.9 KB a workgroup in all, which seven would fit; registers leave room for five.)
  extern __shared__ __align__(16) unsigned char s_v[];

  const int tile_idx = (int)blockIdx.y, z = (int)blockIdx.z;
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
  y = as_global(y);
  w = as_global(w);
  v = as_global(v);
  scales = as_global(scales);
  const bool by_pos = PARTIAL || COMP || v_by_pos;
  unsigned char *const s_v2 = s_v + (COMP ? cnt * VLD * 16 : 0);
  int32_t *const s_perm = reinterpret_cast<int32_t *>(s_v + (COMP ? 2 : 1) * cnt * VLD * 16);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, kg = lane >> 4;
  const uint32_t o_wave = blockIdx.x * (uint32_t)EXP_BN + (uint32_t)(wave * EXP_WN);
  const int rk = min(r, kmax);  // rank columns the narrow operand really has (bgmv_impl.cuh:167,186)

  // ---- everything that depends only on the record: token indices, pool rows of the B fragments, scale, v rows by position
  const int my_perm = perm[pos0 + min(tid, cnt - 1)];
  const float scale = Tr::to_float(scales[ad]);
  const SmallPool pool = {w, a_loc, (uint32_t)h_n_loc, (uint32_t)w_rows, (uint32_t)h_out, inv_h_out, (uint32_t)(astart + r * slot), r, rk};
  SmallRows<KB, WIDE> rows, rows2;
  small_look_up<KB, WIDE>(pool, o_wave, lane, rows);
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
  // The v rows go through LDS, whole lines, once per workgroup: loaded as MFMA operands by every wave they are as many bytes as
  // the y rows, in a pattern that a compute unit takes 64 cycles an instruction for.  16-byte chunk c of row `row` stands at chunk
  // row * VLD + c (VLD odd: 16 rows of one chunk spread over the banks), zeros from rank rk on.
  // A thread's chunks are requested EXP_V_BATCH at a time, `put` writes them.
  const int n_chunks = cnt * VC;
  auto v_request = [&](int e0, const uint16_t *src, int rkk, bool pos, u32x4 (&q)[EXP_V_BATCH]) {
#pragma unroll
    for (int u = 0; u < EXP_V_BATCH; ++u) {
      const int e = e0 + u * 256 + tid;
      if (e0 + u * 256 + wave * 64 >= n_chunks) break;   // wave-uniform
      const int row = min(e / VC, cnt - 1), j0 = (e % VC) * 8;
      if constexpr (PARTIAL) {
        // split-K partials of the shrink: four chunks are requested before any is consumed, summed in chunk order and
        // rounded to T once
        u32x4 f[1];
        small_v_partials<T, 1>(as_global(p.partial) + z * p.partial_tstride + (int64_t)pos0 * p.rp, (uint32_t)(row * p.rp + (j0 < rkk ? j0 : 0)),
                               (int64_t)p.T * p.rp, p.ksplit, 8, 0, f);
        q[u] = j0 < rkk ? f[0] : u32x4{0, 0, 0, 0};
      } else {
        const uint32_t vrow = pos ? (uint32_t)(pos0 + row) : (uint32_t)s_perm[row];
        q[u] = load16(small_source(j0 < rkk, src + (uint64_t)vrow * (uint64_t)v_stride + j0));
      }
    }
  };
  auto v_put = [&](int e0, unsigned char *dst, const u32x4 (&q)[EXP_V_BATCH]) {
#pragma unroll
    for (int u = 0; u < EXP_V_BATCH; ++u) {
      const int e = e0 + u * 256 + tid;
      if (e0 + u * 256 + wave * 64 >= n_chunks) break;
      if (e < n_chunks) *reinterpret_cast<u32x4 *>(dst + ((e / VC) * VLD + e % VC) * 16) = q[u];
    }
  };
  u32x4 q[EXP_V_BATCH];
  if (by_pos) {
    for (int e0 = 0; e0 < n_chunks; e0 += 256 * EXP_V_BATCH) {
      v_request(e0, v + z * v_tstride, rk, true, q);
      v_put(e0, s_v, q);
    }
    if constexpr (COMP)   // the same positions' rows of the merged adapter's matrix
      for (int e0 = 0; e0 < n_chunks; e0 += 256 * EXP_V_BATCH) {
        v_request(e0, v + v_tstride, pool2.rk, true, q);
        v_put(e0, s_v2, q);
      }
  }
  if (tid < cnt) s_perm[tid] = my_perm;
  // This barrier drains the loads above, which everything below needs anyway.  None may follow the bulk loads below: a barrier
  // waits for all outstanding global loads and would serialise the B and y traffic into separate round trips.
  __syncthreads();

  // rows of the caller's matrix are found through the tokens: requested in front of B and y, written behind
  if (!by_pos) v_request(0, v, rk, false, q);

  // row-major roles for the y read-modify-write: 8 lanes x 16 B cover one token row of the wave's
  // 64 outputs; a wave covers 8 rows per access, two accesses per 16-token block.  A row or column that is not there is the
  // tile's last row or the row's first column: read, and not stored.
  const int rr0 = lane >> 3, c8 = (lane & 7) * 8;
  const bool ocol_ok = o_wave + c8 < (uint32_t)h_out;
  uint16_t *const ycol = y + (ocol_ok ? o_wave + c8 : 0u);
  u32x4 yv[MBU][2];
  uint16_t *yp[MBU][2];
  auto load_y = [&](int mb0) {
    int t[MBU][2];
#pragma unroll
    for (int b = 0; b < MBU; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) t[b][h] = s_perm[min((mb0 + b) * 16 + rr0 + 8 * h, cnt - 1)];
#pragma unroll
    for (int b = 0; b < MBU; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        yp[b][h] = ycol + (uint64_t)(uint32_t)t[b][h] * (uint32_t)h_out;
        yv[b][h] = ONCE ? load16_once(yp[b][h]) : load16(yp[b][h]);
      }
  };
  u32x4 bfrag[4 * KB], bfrag2[COMP ? 4 * KB : 1];
  small_load_b<KB, WIDE, true>(pool, lane, rows, bfrag);
  if constexpr (COMP) small_load_b<KB, WIDE, true>(pool2, lane, rows2, bfrag2);
  load_y(0);
  requested();
  if (!by_pos) {
    v_put(0, s_v, q);
    for (int e0 = 256 * EXP_V_BATCH; e0 < n_chunks; e0 += 256 * EXP_V_BATCH) {
      v_request(e0, v, rk, false, q);
      v_put(e0, s_v, q);
    }
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
    requested();
  }
  if (o_wave >= (uint32_t)h_out) return;

  // Two 16-token blocks per iteration: their y rows are all requested before either
  // block is consumed, so an iteration costs one memory round trip for 32 tokens.
  for (int mb0 = 0;;) {
#pragma unroll
    for (int b = 0; b < MBU; ++b) {
      const int row0 = (mb0 + b) * 16;
      if (b > 0 && row0 >= cnt) break;   // workgroup-uniform
      // ---- delta block through the matrix cores, output by token (expand_core.h: a lane has 16 consecutive outputs of token
      // lrow), turned through LDS into rows and added to y
      auto add = [&](const unsigned char *vs, const u32x4 (&bf)[4 * KB], float sc, bool last) {
        u32x4 vf[KB];
        const unsigned char *const vrow = vs + (min(row0 + lrow, cnt - 1) * VLD + kg) * 16;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) vf[kb] = *reinterpret_cast<const u32x4 *>(vrow + kb * 64);
        f32x4 acc[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int nb = 0; nb < 4; ++nb) acc[nb] = Tr::mfma(as<vec8>(bf[nb * KB + kb]), as<vec8>(vf[kb]), acc[nb]);
        // Eight tokens at a time.  stage[wave] is private to this wave and a wave's LDS operations execute in order, so only
        // the compiler has to be kept from reordering the reads below over the writes above.
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if ((lrow >> 3) == h) {
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) *reinterpret_cast<f32x4 *>(&stage[wave][lrow & 7][kg * 16 + nb * 4]) = acc[nb];
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
          const float *srow = &stage[wave][rr0][c8];
          float f[8];
          unpack8<T>(yv[b][h], f);
#pragma unroll
          for (int i = 0; i < 8; ++i) f[i] += sc * srow[i];
          yv[b][h] = pack8<T>(f);
          if (last && ocol_ok && row0 + rr0 + 8 * h < cnt) {
            if (THROUGH) store16_through(yp[b][h], yv[b][h]);
            else store16(yp[b][h], yv[b][h]);
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
      };
      if (!COMP || rk > 0) add(s_v, bfrag, scale, !COMP);
      if constexpr (COMP) add(s_v2, bfrag2, scale2, true);
    }
    mb0 += MBU;
    if (mb0 * 16 >= cnt) break;
    load_y(mb0);
  }
}

// Tiles of 16 tokens (decode batches).  Four independent waves of 64 outputs each: no LDS, no barrier (expand_core.h has
// the loads and the product, and what it measured).  Grid: (column chunks, tiles, targets).
// (Two or four column chunks a workgroup, all their loads in flight together, lose wherever the narrow operand is finished: 512
// tokens, q+k+v at rank 16 26.1 / 27.5 us with its shrink, one target of 256 tokens, 11008 columns 8.6 / 9.6, ranks 8-64, gate+up
// of 13824 columns 25.2 / 27.4.)
constexpr int small_min_waves(int kb, bool wide, bool comp) {   // as many as do without spills
  return comp ? (kb <= 1 ? 7 : 1) : kb <= 1 ? 8 : kb == 2 ? (wide ? 6 : 5) : (wide ? 4 : 3);
}
// THROUGH: y is written through (expand_core.h), up to rank 64.  A form of its own here as well: the exchange of halves behind a flag costs the
// others 0.12 to 0.18 us a launch (5 tokens of rank 16, two targets of 14336 columns 3.62 / 3.50 us, one of 4096 4.48 / 4.30).
template <typename T, int KB, bool WIDE, bool PARTIAL, bool COMP, bool THROUGH>
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
  if constexpr (THROUGH) small_store_y_through(yy, lane, cnt);
  else small_store_y(yy);
}

template <typename T, int KB>
int launch_small_kb(hipStream_t st, const ExpandArgs &a, int64_t tiles) {
  // an index without entries: the kernel reads one all the same, and drops it
  const int64_t *a_loc = a.pool.a_loc_len > 0 ? a.pool.a_loc : reinterpret_cast<const int64_t *>(a.plan + a.off_perm);
#define MLORA_SMALL_FORM(WIDE, PARTIAL, COMP, THROUGH)                                                           \
  hipLaunchKernelGGL((expand_small_kernel<T, KB, WIDE, PARTIAL, COMP, THROUGH>), grid, dim3(256), 0, st, records, \
                     a.plan + a.off_perm, a_loc, (int)a.pool.a_loc_len, a.h_out, a)
#define MLORA_SMALL(WIDE, PARTIAL, COMP)                                                          \
  if (KB < 4 && a.through) MLORA_SMALL_FORM(WIDE, PARTIAL, COMP, (KB < 4));                       \
  else MLORA_SMALL_FORM(WIDE, PARTIAL, COMP, false)
#define MLORA_SMALL_WIDTH(PARTIAL, COMP)                                           \
  if (KB > 0 && a.h_out >= SMALL_WIDE) { MLORA_SMALL((KB > 0), PARTIAL, COMP); }   \
  else { MLORA_SMALL(false, PARTIAL, COMP); }
  // Exactly as many workgroups as there are records: what stands behind the last one is no record (the words of the one-launch
  // op do, and a call of that kind leaves them non-zero).  More tiles than a grid's y takes (a million tokens) are several launches.
  for (int64_t t0 = 0; t0 < tiles; t0 += MAX_GRID_TILES) {
    const int32_t *records = a.plan + a.off_tiles + t0 * TILE_WORDS;
    const dim3 grid((unsigned)a.n_ochunks, (unsigned)(tiles - t0 < MAX_GRID_TILES ? tiles - t0 : MAX_GRID_TILES), (unsigned)a.n_targets);
    if (a.compensate) { MLORA_SMALL_WIDTH(false, true); }
    else if (a.partial) { MLORA_SMALL_WIDTH(true, false); }
    else { MLORA_SMALL_WIDTH(false, false); }
  }
#undef MLORA_SMALL_WIDTH
#undef MLORA_SMALL
#undef MLORA_SMALL_FORM
  return check_launch("expand_small_kernel");
}

template <typename T>
int launch_small_t(hipStream_t st, const ExpandArgs &a, int max_rank, int64_t tiles) {
  if (max_rank <= 16) return launch_small_kb<T, 0>(st, a, tiles);
  if (max_rank <= 32) return launch_small_kb<T, 1>(st, a, tiles);
  if (max_rank <= 64) return launch_small_kb<T, 2>(st, a, tiles);
  return launch_small_kb<T, 4>(st, a, tiles);
}

template <typename T, int KB>
int launch_expand_kb(hipStream_t st, const ExpandArgs &a, int bm, int64_t tiles) {
  // an index without entries: the kernel reads one all the same, and drops it
  const int64_t *a_loc = a.pool.a_loc_len > 0 ? a.pool.a_loc : reinterpret_cast<const int64_t *>(a.plan + a.off_perm);
  const int lds = bm * ((a.compensate ? 2 : 1) * expand_v_chunks(KB) * 16 + 4);
  const bool once = a.through && write_through(a, L2_BYTES);
#define MLORA_EXPAND_FORM(WIDE, PARTIAL, COMP, THROUGH, ONCE)                                                         \
  hipLaunchKernelGGL((expand_kernel<T, KB, WIDE, PARTIAL, COMP, THROUGH, ONCE>), grid, dim3(256), lds, st, records,   \
                     a.plan + a.off_perm, a_loc, (int)a.pool.a_loc_len, a.h_out, a)
#define MLORA_EXPAND(WIDE, PARTIAL, COMP)                                                             \
  if (!COMP && !PARTIAL && once) MLORA_EXPAND_FORM(WIDE, PARTIAL, COMP, !COMP, (!COMP && !PARTIAL));  \
  else if (!COMP && a.through) MLORA_EXPAND_FORM(WIDE, PARTIAL, COMP, !COMP, false);                  \
  else MLORA_EXPAND_FORM(WIDE, PARTIAL, COMP, false, false)
#define MLORA_EXPAND_WIDTH(PARTIAL, COMP)                     \
  if (a.h_out >= SMALL_WIDE) { MLORA_EXPAND(true, PARTIAL, COMP); } \
  else { MLORA_EXPAND(false, PARTIAL, COMP); }
  for (int64_t t0 = 0; t0 < tiles; t0 += MAX_GRID_TILES) {
    const int32_t *records = a.plan + a.off_tiles + t0 * TILE_WORDS;
    const dim3 grid((unsigned)a.n_ochunks, (unsigned)(tiles - t0 < MAX_GRID_TILES ? tiles - t0 : MAX_GRID_TILES), (unsigned)a.n_targets);
    if (a.compensate) { MLORA_EXPAND_WIDTH(false, true); }
    else if (a.partial) { MLORA_EXPAND_WIDTH(true, false); }
    else { MLORA_EXPAND_WIDTH(false, false); }
  }
#undef MLORA_EXPAND_WIDTH
#undef MLORA_EXPAND
#undef MLORA_EXPAND_FORM
  return check_launch("expand_kernel");
}

template <typename T>
int launch_expand_t(hipStream_t st, const ExpandArgs &a, int max_rank, int bm, int64_t tiles) {
  if (max_rank <= 32) return launch_expand_kb<T, 1>(st, a, bm, tiles);
  if (max_rank <= 64) return launch_expand_kb<T, 2>(st, a, bm, tiles);
  return launch_expand_kb<T, 4>(st, a, bm, tiles);
}

}  // namespace

int launch_expand(hipStream_t st, const ExpandArgs &args, int max_rank, int64_t grid_tiles, int bm_expand, mlora_dtype dt) {
  if (grid_tiles <= 0) return MLORA_OK;
  ExpandArgs a = args;
  a.through = write_through(a, THROUGH_BYTES);
  if (bm_expand == 16)
    return dt == MLORA_F16 ? launch_small_t<_Float16>(st, a, max_rank, grid_tiles) : launch_small_t<__bf16>(st, a, max_rank, grid_tiles);
  return dt == MLORA_F16 ? launch_expand_t<_Float16>(st, a, max_rank, bm_expand, grid_tiles)
                         : launch_expand_t<__bf16>(st, a, max_rank, bm_expand, grid_tiles);
}

int expand_bn() { return EXP_BN; }

}  // namespace mlora
