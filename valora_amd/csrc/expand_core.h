// Operands in lane order: the B fragments and the summed split-K partials, loaded as whole lines and turned through LDS.
// Used by the column-looping expand (csrc/expand.hip) and, for B, by the merge (csrc/merge.hip).
#pragma once

#include "kernel_common.h"

namespace mlora {

// v_mfma_f32_16x16x32 wants lane (column = lane%16, kgroup = lane/16) to hold 8 consecutive rank elements of one
// output.  In the pool an output's r rank elements are consecutive, so lanes that load that way sit 2*r bytes apart and
// fill the load instructions badly (half of the lanes masked at rank 16, another 128-byte line per lane from rank 64 on,
// which costs a compute unit some 64 cycles per instruction instead of 16).  A wave's 64 outputs are one run of 128*r
// bytes, so the column-looping expand, whose workgroups fill the device several times over, loads them in lane order
// -- whole lines, nothing masked -- and turns them into operands through a piece of LDS of the wave's own (no barrier:
// a wave's LDS accesses run in order; units XOR-swizzled so that the 16-byte reads, r/8 units apart, spread over the
// banks).  Direct / lane order with a finished v, cold layers: 256 tokens over 64 adapters of rank 16, two targets of 3072
// columns 7.8 / 6.6 us, q+k+v of 4096 10.9 / 11.2, gate+up of 11008 18.0 / 17.0; of rank 64 17.6 / 15.6, 25.2 / 26.5 and
// 41.6 / 41.8; 77 tokens over ranks 8-64, gate+up of 13824 17.7 / 17.0; a decode pass of those over eight layers 701 / 686.
// (Above rank 64, and in the other expand kernels, operands are loaded directly: there the registers and the turn cost
// more than the instructions, 6.2 -> 6.6 us for one decode target, 26 -> 31 us for a 6749-token prefill at rank 32.)
constexpr int B_TURN_BYTES = 4096;   // LDS of a wave's turn: 256 units of 16 bytes
constexpr int B_OUTS = 64;           // outputs per wave

__device__ __forceinline__ uint32_t b_swizzle(uint32_t q) { return q ^ (((q >> 3) ^ (q >> 6)) & 7u); }

// Units an output has in the turn.  KB is the class of the narrow operand (up to 32 * KB columns), r the adapter's rank.
// WIDER: r may be above the class.  What lies beyond the class meets no column of the operand: it is neither loaded nor
// turned, so that a pass has at most 256 units whatever the rank.
template <int KB, bool WIDER>
__device__ __forceinline__ constexpr uint32_t b_rank_units(uint32_t r) {
  return WIDER && r > 32u * KB ? 4u * KB : r >> 3;
}
static_assert(B_OUTS * 4 * 16 <= B_TURN_BYTES, "a pass, B_OUTS / KB outputs of up to 4 * KB units, fits the turn");

// A wave's B operands are turned in KB passes of B_OUTS / KB outputs, up to 4 instructions (256 units) each.
// A lane's own part of the flat element its units start at.
template <int KB, bool WIDER>
__device__ __forceinline__ uint32_t b_lane(int lane, uint32_t r) {
  // (outputs of more units than the class uses lie apart)
  return (uint32_t)lane * 8u + (WIDER ? (uint32_t)lane / (4u * KB) * (r - 8u * b_rank_units<KB, WIDER>(r)) : 0u);
}
// The flat element a lane's unit i of pass p starts at, `own` from b_lane, `first` that of the wave's first output; false:
// no such unit.
template <int KB, bool WIDER>
__device__ __forceinline__ bool b_unit(int p, int i, int lane, uint32_t own, uint32_t r, uint32_t first, uint32_t &flat) {
  constexpr uint32_t OUTS = B_OUTS / KB;
  const uint32_t units = b_rank_units<KB, WIDER>(r);
  flat = first + (uint32_t)p * OUTS * r + (uint32_t)i * (512u + (WIDER ? 16u / KB * (r - 8u * units) : 0u)) + own;
  return (uint32_t)(i * 64 + lane) < OUTS * units;
}
// wave-uniform: whether instruction i of a pass has any unit
template <int KB, bool WIDER>
__device__ __forceinline__ bool b_any(int i, uint32_t r) {
  return (uint32_t)(i * 64) < (B_OUTS / KB) * b_rank_units<KB, WIDER>(r);
}

// raw[p][i] as loaded -> bfrag[nb][kb] = B^T[o = nb*16 + lane%16][kb*32 + (lane/16)*8 .. + 8), zero from rank rk on
// (rk <= r, rk <= 32 * KB).
// `turn`: B_TURN_BYTES of LDS of this wave.
template <int KB, bool WIDER>
__device__ __forceinline__ void b_turn(const u32x4 (&raw)[KB][4], u32x4 (&bfrag)[4][KB], uint32_t r, int rk, int lane,
                                       unsigned char *turn) {
  const uint32_t rq = b_rank_units<KB, WIDER>(r);
  const int lrow = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int p = 0; p < KB; ++p) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (b_any<KB, WIDER>(i, r)) *reinterpret_cast<u32x4 *>(turn + b_swizzle((uint32_t)(i * 64 + lane)) * 16u) = raw[p][i];
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

// The v operand of one 16-token block from the split-K partials: `part` is the block's first row in chunk 0, rows of
// rp floats one after the other, chunks `sstride` floats apart.  The block is one run of 64*rp bytes per chunk, loaded
// in lane order; every lane adds up its own four columns over the chunks in index order, rounds once, and the rows
// are turned into operands through LDS like B above.  Rows from cnt on and ranks from rk on are zero.  Loaded row by row /
// so, B directly in both: 256 tokens over 64 adapters, q+k+v of 4096 columns at rank 16 12.4 / 11.8 us, at rank 64 28.4 /
// 26.6, one target at rank 32 8.1 / 7.7; 512 tokens over 128 adapters of rank 128, one target 31.4 / 28.8.
template <typename T, int KB>
__device__ __forceinline__ void v_from_partials(const float *part, int64_t sstride, int ksplit, int rp, int cnt, int rk,
                                                int lane, unsigned char *turn, u32x4 (&vfrag)[KB]) {
  constexpr int G = 2 * KB;                              // groups of 64 units of four floats; rp <= 32 * KB
  const int lrow = lane & 15, kg = lane >> 4;
  f32x4 sum[G];
#pragma unroll
  for (int g = 0; g < G; ++g) sum[g] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int n_units = cnt * (rp >> 2);                   // rows in use
  constexpr int BATCH = 4 / KB;                          // chunks whose loads are in flight together
  for (int s0 = 0; s0 < ksplit; s0 += BATCH) {
    f32x4 q[BATCH][G];
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
#pragma unroll
      for (int g = 0; g < G; ++g)
        q[u][g] = (s0 + u < ksplit && g * 64 + lane < n_units)
                      ? *reinterpret_cast<const f32x4 *>(part + (int64_t)(s0 + u) * sstride + (g * 64 + lane) * 4)
                      : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
#pragma unroll
      for (int g = 0; g < G; ++g) sum[g] += q[u][g];
  }
  using Tr = Traits<T>;
#pragma unroll
  for (int g = 0; g < G; ++g)
    if (g * 64 < 4 * rp)
      *reinterpret_cast<uint2 *>(turn + (g * 64 + lane) * 8) =
          uint2{Tr::pack2(sum[g][0], sum[g][1]), Tr::pack2(sum[g][2], sum[g][3])};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int j0 = kb * 32 + kg * 8;
    const bool ok = lrow < cnt && j0 < rk;
    const u32x4 got = *reinterpret_cast<const u32x4 *>(turn + (lrow * rp + (ok ? j0 : 0)) * 2);
    vfrag[kb] = ok ? got : u32x4{0, 0, 0, 0};
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace mlora
