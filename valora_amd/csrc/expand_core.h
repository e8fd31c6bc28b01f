// Operands of the expand: B in lane order, loaded as whole lines and turned through LDS (the merge, csrc/merge.hip), and
// the expand of tiles of at most 16 tokens (csrc/expand.hip, csrc/decode.hip).
#pragma once

#include "kernel_common.h"

namespace mlora {

// ---- B in lane order -------------------------------------------------------------------------------------------------
// v_mfma_f32_16x16x32 wants lane (column = lane%16, kgroup = lane/16) to hold 8 consecutive rank elements of one
// output.  In the pool an output's r rank elements are consecutive, so lanes that load that way sit 2*r bytes apart and
// fill the load instructions badly (half of the lanes masked at rank 16, another 128-byte line per lane from rank 64 on,
// which costs a compute unit some 64 cycles per instruction instead of 16).  A wave's 64 outputs are one run of 128*r
// bytes, so the merge, whose workgroups fill the device several times over, loads them in lane order
// -- whole lines, nothing masked -- and turns them into operands through a piece of LDS of the wave's own (no barrier:
// a wave's LDS accesses run in order; units XOR-swizzled so that the 16-byte reads, r/8 units apart, spread over the
// banks).  (In the expand kernels operands are loaded directly: there the registers and the turn cost more than the
// instructions, 6.2 -> 6.6 us for one decode target, 26 -> 31 us for a 6749-token prefill at rank 32.)
constexpr int B_TURN_BYTES = 4096;   // LDS of a wave's turn: 256 units of 16 bytes
constexpr int B_OUTS = 64;           // outputs per wave

__device__ __forceinline__ uint32_t b_swizzle(uint32_t q) { return q ^ (((q >> 3) ^ (q >> 6)) & 7u); }

// KB is the class of the ranks (up to 32 * KB), r the adapter's rank, r/8 the units of an output.
static_assert(B_OUTS * 4 * 16 <= B_TURN_BYTES, "a pass, B_OUTS / KB outputs of up to 4 * KB units, fits the turn");

// A wave's B operands are turned in KB passes of B_OUTS / KB outputs, up to 4 instructions (256 units) each.
// The flat element a lane's unit i of pass p starts at, `first` that of the wave's first output; false: no such unit.
template <int KB>
__device__ __forceinline__ bool b_unit(int p, int i, int lane, uint32_t r, uint32_t first, uint32_t &flat) {
  constexpr uint32_t OUTS = B_OUTS / KB;
  flat = first + (uint32_t)p * OUTS * r + (uint32_t)(i * 64 + lane) * 8u;
  return (uint32_t)(i * 64 + lane) < OUTS * (r >> 3);
}
// wave-uniform: whether instruction i of a pass has any unit
template <int KB>
__device__ __forceinline__ bool b_any(int i, uint32_t r) { return (uint32_t)(i * 64) < (B_OUTS / KB) * (r >> 3); }

// raw[p][i] as loaded -> bfrag[nb][kb] = B^T[o = nb*16 + lane%16][kb*32 + (lane/16)*8 .. + 8), zero from rank rk on
// (rk <= r <= 32 * KB).
// `turn`: B_TURN_BYTES of LDS of this wave.
template <int KB>
__device__ __forceinline__ void b_turn(const u32x4 (&raw)[KB][4], u32x4 (&bfrag)[4][KB], uint32_t r, int rk, int lane,
                                       unsigned char *turn) {
  const uint32_t rq = r >> 3;
  const int lrow = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int p = 0; p < KB; ++p) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (b_any<KB>(i, r)) *reinterpret_cast<u32x4 *>(turn + b_swizzle((uint32_t)(i * 64 + lane)) * 16u) = raw[p][i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int n = 0; n < 4 / KB; ++n)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const uint32_t c = (uint32_t)(kb * 4 + kg);
        const bool ok = (int)(c * 8u) < rk;
        const uint32_t q = (uint32_t)(n * 16 + lrow) * rq + (ok ? c : 0u);
        const u32x4 got = *reinterpret_cast<const u32x4 *>(turn + b_swizzle(q) * 16u);
        bfrag[p * (4 / KB) + n][kb] = ok ? got : u32x4{0, 0, 0, 0};
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- tiles of at most 16 tokens ---------------------------------------------------------------------------------------
// What the expand of a decode batch waits for is its own instructions: a wave has a few KB of B and y, and address set-up,
// masks and the turn of the result used to be 390 vector instructions (2100 cycles a wave, 3.5 us of the 5.9 us of 1024
// workgroups); here they are 150.
//
// The product is formed the other way round than in the expand of tall tiles: D = B^T v^T, so that a lane ends up with
// outputs of one token (column = token = lane%16, rows 4*(lane/16) + i = outputs).  Which output a row stands for is free
// to choose: row m of fragment nb is output 16*(m/4) + 4*nb + m%4 of the wave's 64, so a lane's four fragments hold 16
// consecutive outputs of its token, which it updates in y itself, 32 bytes at once: no turn through LDS, no LDS and no
// barrier at all.  Every element is the same sum in the same order either way: same bits.
//
// One target, cold layers, before (expand_kernel, or a loop over two column chunks for big grids) / now: 256 tokens over 64 adapters of rank 16,
// 4096 columns 5.8 / 5.0 us, 11008 columns 10.0 / 8.6; one token 3.1 / 2.2; 77 tokens over ranks 8-64, 5120 columns 6.8 / 5.9;
// 256 tokens over 64 adapters of rank 64 11.3 / 9.9; 100 over 16 of rank 128, 3072 columns 7.9 / 6.4; 512 over 128 of rank 128
// 30.4 / 30.1.
//
// KB: 32-wide rank blocks of the narrow operand, 0 where it has at most 16 columns.  Half of an operand would be
// zeros then, so one load fetches two fragments, the second one with lanes 32-63, and a swap of lane halves puts
// that one in its place.
template <int KB>
struct SmallB {
  static constexpr int FRAG_KB = KB ? KB : 1;         // operands per fragment
  static constexpr int LOADS = KB ? 4 * KB : 2;
  // what a lane fetches: LOADS units of 8 rank elements, unit i at flat element first + step(i) of the slot's B
  static __device__ __forceinline__ uint32_t lane_output(int lane) {   // of the first unit, within the wave's 64
    const int m = lane & 15;
    return KB ? (uint32_t)((m >> 2) * 16 + (m & 3)) : (uint32_t)((m >> 2) * 8 + (m & 3) + (lane >> 5) * 4);
  }
  static __device__ __forceinline__ int lane_rank(int lane) { return ((lane >> 4) & (KB ? 3 : 1)) * 8; }
  static __device__ __forceinline__ uint32_t step(int i, int r) {
    return KB ? (uint32_t)((i / FRAG_KB) * 4 * r + (i % FRAG_KB) * 32) : (uint32_t)(i * 32 * r);
  }
  static __device__ __forceinline__ bool in_rank(int i, int lane, int rk) { return lane_rank(lane) + (KB ? i % FRAG_KB * 32 : 0) < rk; }
};

// The pool rows a lane's units lie in, as looked up.  WIDE: outputs so wide that the units, which start at most
// 12 * r + 32 * (KB - 1) elements apart, lie in two neighbouring rows whatever the rank; below that every unit has a look-up of its own.
constexpr int SMALL_WIDE = 12 * MAX_RANK + 96;
template <int KB, bool WIDE>
struct SmallRows {
  static constexpr int N = WIDE ? 2 : SmallB<KB>::LOADS;
  uint32_t off[WIDE ? 1 : N];   // element of its row the first (every) unit starts at
  int64_t row[N];
  bool ok[N];
};
// Where everything is that the look-ups and loads of one target need
struct SmallPool {
  const uint16_t *w;
  const int64_t *a_loc;
  uint32_t n_loc, w_rows, h_out;   // a_loc has at least one entry
  float inv_h_out;
  uint32_t base;                   // index entry of the slot's first row (negative: no entry, as unsigned)
  int r, rk;                       // the adapter's rank and the columns of it the narrow operand has
};
template <int KB, bool WIDE>
__device__ __forceinline__ void small_look_up(const SmallPool &p, uint32_t o_wave, int lane, SmallRows<KB, WIDE> &s) {
  using B = SmallB<KB>;
  const uint32_t first = (o_wave + B::lane_output(lane)) * (uint32_t)p.r + (uint32_t)B::lane_rank(lane);   // < 2^16 * 2^7
  uint32_t bin;
#pragma unroll
  for (int k = 0; k < SmallRows<KB, WIDE>::N; ++k) {
    if (!WIDE) divmod24(first + B::step(k, p.r), p.h_out, p.inv_h_out, bin, s.off[WIDE ? 0 : k]);
    else if (k == 0) divmod24(first, p.h_out, p.inv_h_out, bin, s.off[0]);
    const uint32_t idx = p.base + bin + (WIDE ? k : 0);
    s.ok[k] = idx < p.n_loc;
    s.row[k] = p.a_loc[s.ok[k] ? idx : 0u];
  }
}
// What a lane without anything to fetch reads instead.  (A masked load takes two exec changes, a branch and four moves
// for the zeros; a choice between two addresses takes two moves, and nothing stands between one load and the next.)
__device__ const __align__(128) uint16_t g_small_zeros[64] = {};
__device__ __forceinline__ const uint16_t *small_source(bool ok, const void *src) {
  return as_global(reinterpret_cast<const uint16_t *>(ok ? src : static_cast<const void *>(g_small_zeros)));
}
// Requests the lane's units; units without a pool row are zero, those beyond the narrow operand's columns are zero with IN_RANK,
// else whatever stands there (small_product drops them).
template <int KB, bool WIDE, bool IN_RANK = false>
__device__ __forceinline__ void small_load_b(const SmallPool &p, int lane, const SmallRows<KB, WIDE> &s, u32x4 (&raw)[SmallB<KB>::LOADS]) {
  using B = SmallB<KB>;
  constexpr int N = SmallRows<KB, WIDE>::N;
  const char *bp[N];
  bool bok[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    bok[k] = s.ok[k] && (uint64_t)s.row[k] < (uint64_t)p.w_rows;
    bp[k] = reinterpret_cast<const char *>(p.w) + (uint64_t)(uint32_t)s.row[k] * (p.h_out * 2u);
  }
#pragma unroll
  for (int i = 0; i < B::LOADS; ++i) {
    const char *src;
    bool ok;
    if constexpr (WIDE) {
      const uint32_t at = s.off[0] + B::step(i, p.r);
      const bool second = at >= p.h_out;
      src = (second ? bp[1] : bp[0]) + (at - (second ? p.h_out : 0u)) * 2u;
      ok = (second && bok[1]) || (!second && bok[0]);
    } else {
      src = bp[i] + s.off[i] * 2u;
      ok = bok[i];
    }
    raw[i] = load16(small_source(ok && (!IN_RANK || B::in_rank(i, lane, p.rk)), src));
  }
}
// acc[nb] = fragment nb of B^T times v^T; units beyond the operand's columns count as zero.  (Masked here and not at the load:
// the address of a unit that is not there and needs no pool row is as good as another, and a choice less per load; 512 tokens
// over 128 adapters of rank 128, shrink and expand 62.7 -> 61.1 us, rank 8, gate+up of 8192 columns 27.1 -> 26.5.)
template <typename T, int KB>
__device__ __forceinline__ void small_product(const u32x4 (&raw)[SmallB<KB>::LOADS], const u32x4 (&vfrag)[SmallB<KB>::FRAG_KB], int rk, int lane,
                                              f32x4 (&acc)[4]) {
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (KB == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool in = SmallB<KB>::in_rank(i, lane, rk);
      u32x4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // lanes 32-63 of what was loaded change places with lanes 0-31 of a zero
        const auto sw = __builtin_amdgcn_permlane32_swap(in ? raw[i][e] : 0u, 0u, false, false);
        lo[e] = sw[0];
        hi[e] = sw[1];
      }
      acc[2 * i] = Tr::mfma(as<vec8>(lo), as<vec8>(vfrag[0]), acc[2 * i]);
      acc[2 * i + 1] = Tr::mfma(as<vec8>(hi), as<vec8>(vfrag[0]), acc[2 * i + 1]);
    }
  } else {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        if (kb * 32 < rk) {
          const bool in = SmallB<KB>::in_rank(kb, lane, rk);
          const u32x4 b = raw[nb * KB + kb];
          acc[nb] = Tr::mfma(as<vec8>(in ? b : u32x4{0, 0, 0, 0}), as<vec8>(vfrag[kb]), acc[nb]);
        }
  }
}
// The narrow operand of the lane's token from split-K partials: its row is `row` floats behind `tile` (the same for all
// lanes), chunks `stride` floats apart.  Four chunks are requested before any is used (the last one again where there are
// fewer: what is loaded under a condition the compiler loads where it is used, one round trip each), summed in index order
// and rounded once.
template <typename T, int KB>
__device__ __forceinline__ void small_v_partials(const float *tile, uint32_t row, int64_t stride, int ksplit, int rk, int lane,
                                                 u32x4 (&vfrag)[SmallB<KB>::FRAG_KB]) {
#pragma unroll
  for (int kb = 0; kb < SmallB<KB>::FRAG_KB; ++kb) {
    const int j0 = kb * 32 + (lane >> 4) * 8;
    const bool ok = j0 < rk;
    const uint32_t at = (row + (uint32_t)(ok ? j0 : 0)) * 4u;
    float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const char *chunk = reinterpret_cast<const char *>(tile);
    auto add_four = [&](int s0) {
      f32x4 lo[4], hi[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const f32x4 *src = reinterpret_cast<const f32x4 *>(chunk + at);
        lo[u] = src[0];
        hi[u] = src[1];
        chunk = next_chunk(chunk, s0 + u + 1 < ksplit, stride * 4);
      }
      requested();
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s0 + u < ksplit) {   // wave-uniform
#pragma unroll
          for (int i = 0; i < 4; ++i) { f[i] += lo[u][i]; f[4 + i] += hi[u][i]; }
        }
    };
    // (the first four outside the loop: a loop's loads wait for whatever was requested before it)
    add_four(0);
    for (int s0 = 4; s0 < ksplit; s0 += 4) add_four(s0);
    const u32x4 v = pack8<T>(f);
    vfrag[kb] = ok ? v : u32x4{0, 0, 0, 0};
  }
}
// Bytes of y from which a launch writes it through (store16_through).  Cold layers, whole op, 140 shapes: tall tiles (4.8 MB of y and more)
// 0.95 to 0.99 of the time, 1.01 at worst; 16-token tiles of two launches up to rank 64 0.95 to 0.99 from 2.5 MB on, 0.98 to 1.02 at 1 to 2 MB; one
// launch 0.91 to 0.98 from 4.7 MB on (1201 tokens of rank 16, two targets of 8192 columns 26.9 / 24.7 us), 1.00 at 1 to 2.5 MB, and 1.05 for
// a few tokens, where the way to memory is longer than the write-back of what little there is.
constexpr int64_t THROUGH_BYTES = (int64_t)2 << 20, THROUGH_BYTES_ONE_LAUNCH = (int64_t)3 << 20;
// Either only in rows of whole 128-byte lines: a line that two waves store a piece of each goes to memory twice (6700 tokens of rank 64, 4128
// and 8224 columns, a pass of two layers 804 us without, 922 with).  Not in 16-token tiles above rank 64 (csrc/expand.hip), which read
// much more than they write (512 tokens over 128 adapters of rank 128, q+k+v 79.2 / 80.4 us, and 80.0 with the choice alone).  Nor in
// tall tiles of compensations: the merged adapter's tokens are not written, most of the batch in earnest, and the host does not know how many they
// are.  A pass, plain / through: 2817 tokens of rank 128, 2 of them not the merged adapter's 505 / 512 us, 737 of them 665 / 676; 6368 over
// ranks 16-64, 466 751 / 749, 2657 1073 / 1066.  In 16-token tiles up to rank 64 it pays there as well, whatever their number, from half as
// many bytes on: 918 tokens over ranks 16-64, 306 not the merged adapter's 557 / 542, 1100 of rank 32, 958 of them 677 / 654 and 39 of them
// 354 / 348, 600 of rank 16, 44 of them 268 / 269, 900 of rank 64, 33 of them 401 / 405 (the worst of ten).
// (Tokens without an adapter are counted: of 1000 tokens of rank 16 in one launch, half of them without, a pass of 8 layers 236 / 226, 95 %
// of them 155 / 159.)
inline int write_through(const ExpandArgs &a, int64_t least) {
  uintptr_t ends = 0;
  for (int z = 0; z < a.n_targets; ++z) ends |= reinterpret_cast<uintptr_t>(a.ys[z]);
  return (int64_t)(a.compensate ? a.T / 2 : a.T) * a.h_out * a.n_targets * 2 >= least && !(a.h_out & 63) && !(ends & 127u);
}
// The lane's outputs of y: 16 from o_wave + 16 * (lane / 16) on, in two 16-byte halves.
template <int KB>
struct SmallY {
  u32x4 v[2];
  uint16_t *p;
  bool ok[2];
};
template <int KB>
__device__ __forceinline__ void small_load_y(SmallY<KB> &s, uint16_t *y, int tok, bool on, uint32_t o_wave, uint32_t h_out, int lane) {
  const uint32_t o = o_wave + (uint32_t)(lane >> 4) * (KB ? 16u : 8u);
  constexpr uint32_t H = KB ? 8u : 32u;
  s.p = reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(y) + (uint64_t)(uint32_t)tok * (h_out * 2u)) + o;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    s.ok[h] = on && o + H * h < h_out;
    s.v[h] = load16(o + H * h < h_out ? s.p + h * (KB ? 8 : 32) : y);   // (lanes without a token read the first one's row)
  }
}
template <typename T, int KB>
__device__ __forceinline__ void small_add(SmallY<KB> &s, const f32x4 (&acc)[4], float scale) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float f[8];
    unpack8<T>(s.v[h], f);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] += scale * acc[h * 2 + (i >> 2)][i & 3];
    s.v[h] = pack8<T>(f);
  }
}
template <int KB>
__device__ __forceinline__ void small_store_y(const SmallY<KB> &s) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
    if (s.ok[h]) store16(s.p + h * (KB ? 8 : 32), s.v[h]);
}
// The same, written through, where rows are whole lines (write_through) and the wave's outputs are there; cnt: tokens of the tile.  A
// lane's halves lie 16 or 64 bytes apart, so that a store of one half writes pieces of lines.  That is all the same to the L2; on their way
// to memory the lanes of a pair, two tokens of the same columns, exchange a half first: every store then writes whole lines of one token.
template <int KB>
__device__ __forceinline__ void small_store_y_through(const SmallY<KB> &s, int lane, int cnt) {
  constexpr int H = KB ? 8 : 32;
  const int m = lane & 15;
  const bool odd = lane & 1;
  const u32x4 give = odd ? s.v[0] : s.v[1];
  u32x4 got;
#pragma unroll
  for (int i = 0; i < 4; ++i) got[i] = lane_pair(give[i]);
  const uint64_t own = (uint64_t)reinterpret_cast<uintptr_t>(s.p);
  const uint64_t other = (uint64_t)lane_pair((uint32_t)own) | (uint64_t)lane_pair((uint32_t)(own >> 32)) << 32;
  uint16_t *const even_row = reinterpret_cast<uint16_t *>(odd ? other : own) + (odd ? H : 0);
  uint16_t *const odd_row = reinterpret_cast<uint16_t *>(odd ? own : other) + (odd ? H : 0);
  if ((m & ~1) < cnt) store16_through(even_row, odd ? got : s.v[0]);
  if ((m | 1) < cnt) store16_through(odd_row, odd ? s.v[1] : got);
}

}  // namespace mlora
