// Device-side helpers shared by the gfx950 LoRA kernels: 16-byte vector access and the
// per-dtype MFMA / conversion traits.  (The reference's counterpart is the 1300-line
// vec_dtypes.cuh, valora/csrc/bgmv/vec_dtypes.cuh:16-30,754-800; only fp16 and bf16 exist here.)
#pragma once

#include "mlora_internal.h"

namespace mlora {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

template <typename To, typename From>
__device__ __forceinline__ To as(const From &v) {
  static_assert(sizeof(To) == sizeof(From), "size mismatch");
  return __builtin_bit_cast(To, v);
}

// One global_load_dwordx4 / global_store_dwordx4.  Addresses must be 16-byte aligned.
__device__ __forceinline__ u32x4 load16(const uint16_t *p) { return *reinterpret_cast<const u32x4 *>(p); }
constexpr int64_t L2_BYTES = (int64_t)32 << 20;   // what the L2s of the eight XCDs hold together
// The same for what nobody reads again soon: the line is the first to leave the caches.  Only where a wave reads whole lines at once: of a
// line read piece by piece it costs a second fetch (B of the expand: 512 tokens over 128 adapters of rank 128, a pass 839 / 912 us).
__device__ __forceinline__ u32x4 load16_once(const uint16_t *p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)); }
__device__ __forceinline__ void store16(uint16_t *p, u32x4 v) { *reinterpret_cast<u32x4 *>(p) = v; }
// The same, on to memory at once instead of leaving a dirty line in the XCD's L2.  The L2s write their dirty lines back when a
// kernel ends, with nothing else to do: 2.4 us of a launch that updates tens of MB.  Pays for whole 128-byte lines (pieces of
// 16 bytes are written to memory one by one); csrc/expand_core.h has the rule.
__device__ __forceinline__ void store16_through(uint16_t *p, u32x4 v) {
  typedef __attribute__((address_space(1))) u32x4 *GP;
  __builtin_amdgcn_global_store_b128((GP)(uintptr_t)p, v, "agent");
}

// The value of the other lane of a pair (lanes 2i and 2i + 1)
__device__ __forceinline__ uint32_t lane_pair(uint32_t x) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true); }

// A pointer that went through an inline asm operand has lost what the compiler knew about it; telling it again that
// the memory is global keeps its loads and stores on the global path (flat accesses count against two wait counters)
template <typename P>
__device__ __forceinline__ P *as_global(P *p) {
  typedef __attribute__((address_space(1))) P *GP;
  return (P *)(GP)(uintptr_t)p;
}

// wait until at most N vector-memory accesses of this wave are outstanding (they retire in order)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// wait until none of its LDS accesses and scalar loads is outstanding
__device__ __forceinline__ void wait_lgkmcnt0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// loads requested above stay above: the compiler would rather sink them to where they are used
__device__ __forceinline__ void requested() { asm volatile("" ::: "memory"); }
// The next of a row of chunks that are requested together, or the same again: the compiler must not see that it may be the
// same, or it branches around the load, one round trip per chunk.
__device__ __forceinline__ const char *next_chunk(const char *chunk, bool more, int64_t stride) {
  chunk += more ? stride : 0;
  asm volatile("" : "+s"(chunk));
  return as_global(chunk);
}
// q = n / d and rem = n % d for n < 2^24 (exact in fp32) from a reciprocal computed once: the float estimate of
// the quotient is off by at most one.  An integer division by a run-time divisor costs some 35 vector
// instructions, and the kernels' address set-up does several per lane before the first load can be issued.
__device__ __forceinline__ void divmod24(uint32_t n, uint32_t d, float inv_d, uint32_t &q, uint32_t &rem) {
  q = (uint32_t)((float)n * inv_d);
  int32_t m = (int32_t)(n - q * d);
  const bool low = m < 0, high = m >= (int32_t)d;   // (selects: a branch would cost more)
  q += high ? 1u : low ? ~0u : 0u;
  m += low ? (int32_t)d : high ? -(int32_t)d : 0;
  rem = (uint32_t)m;
}

template <typename T>
struct Traits;

template <>
struct Traits<_Float16> {
  using vec8 = f16x8;
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float to_float(uint16_t h) { return (float)as<_Float16>(h); }
  static __device__ __forceinline__ uint16_t from_float(float f) { return as<uint16_t>((_Float16)f); }
  // two values, the first in the low half (one by one: behind a multiply-add either becomes a single mixed-precision
  // FMA that rounds to fp16 at once, where a packed conversion would round the fp32 sum)
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return (uint32_t)from_float(lo) | ((uint32_t)from_float(hi) << 16);
  }
};

template <>
struct Traits<__bf16> {
  using vec8 = bf16x8;
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float to_float(uint16_t h) { return as<float>((uint32_t)h << 16); }
  // Round to nearest even, one v_cvt_pk_bf16_f32 for two values.  (Written out in integer arithmetic the rounding is
  // seven instructions a value, which the kernels that update y or W in place have nothing to hide behind: merging
  // an adapter rounds every weight twice.)
  static __device__ __forceinline__ uint16_t from_float(float f) { return as<uint16_t>((__bf16)f); }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    return as<uint32_t>(__builtin_convertvector((f32x2{lo, hi}), bf16x2));
  }
};

// which of the device's XCDs this wave runs on (bits 3:0 of the XCC_ID hardware register)
__device__ __forceinline__ uint32_t xcd_id() { return (uint32_t)__builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20); }

// 8 packed T values <-> 8 floats
template <typename T>
__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = Traits<T>::to_float((uint16_t)(v[i] & 0xffffu));
    f[2 * i + 1] = Traits<T>::to_float((uint16_t)(v[i] >> 16));
  }
}

template <typename T>
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = Traits<T>::pack2(f[2 * i], f[2 * i + 1]);
  return v;
}

}  // namespace mlora
