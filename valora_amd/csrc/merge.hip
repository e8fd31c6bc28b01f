// Merging one adapter into the base weights and taking it out again, for gfx950:
//
//     W_slot[i, o] = T( W_slot[i, o] +- T( sum_{j<r} A[i, j] * T(B[j, o] * scaling) ) )
//
// for the slots (q, k, v, o) of one layer.  This is the reference's merge_adapter / unmerge_adapter
// (valora/models/peft/lora_single_batch_infer.py:103-149): `b = B * scaling` is a T tensor there,
// `ab = bmm(a, b)` is a T tensor (fp32 accumulation inside the GEMM), and `add_` / `sub_` round once
// more; the three rounding points are kept.  The reference first copies the adapter out of the pool
// into dense [H, r] / [r, H] matrices (:81-98), runs the batched GEMM into a [4, H, H] temporary
// and then updates the four weights; here the pool rows are read in place and W is read and
// written exactly once, so the traffic is 2 * H_in * H_out * sizeof(T) per slot.
//
// Layouts: W is [H_in, H_out] row-major (the transposed weight the reference keeps, x @ W).
// B of a slot is [H_out, r] flat over r pool rows -- K-contiguous for the MFMA, loaded straight
// into registers as in the expand.  A of a slot is r pool rows of H_in elements, i.e. [r, H_in]:
// the MFMA wants 8 consecutive rank elements of ONE input row per lane, so the workgroup's
// [r x tile height] slice of A goes through LDS transposed: a thread loads an 8 x 8 block (8 rank rows, 16 bytes
// each), transposes it in registers and writes eight 16-byte units, which the products read as they are.
//
// Bound by the in-place update of W (268 MB for four 4096 x 4096 slots; an in-place stream runs at 4.4-4.9 TB/s on
// this part) up to rank 32, above that also by the operands a workgroup reads beside its share of W: B once per
// workgroup (in lane order, expand_core.h), A once per 256 columns.  Measured, four 4096 x 4096 slots of bf16 weights,
// before / after transposing A once instead of at every use, reading B in lane order and for several slices, all
// look-ups in one round trip, and rounding to bf16 in hardware: rank 16 63.7 / 56.5 us, rank 64 82.6 / 59.0, rank 128
// 126.4 / 68.8.  Of that the rounding alone takes it to 57.6, 72.1 and 99.9; one slice a workgroup would leave 56.5, 66.3
// and 85.6.
#include "expand_core.h"
#include "kernel_common.h"

namespace mlora {

namespace {

constexpr int MG_BN = 256;        // output columns per workgroup, 64 per wave
// input rows (of W) per slice of A in LDS (16 KB up to rank 64, 32 KB above)
constexpr int merge_bm(int kb) { return kb == 1 ? 256 : 128; }
// Workgroups resident per compute unit: four up to rank 64, two above (the B fragments of rank 128 take 64 registers).
constexpr int merge_resident(int kb) { return kb == 4 ? 2 : 4; }
constexpr int MG_STAGE_LD = 64 + 4;

struct MergeArgs {
  uint16_t *w[MLORA_MAX_TARGETS];
  int slots[MLORA_MAX_TARGETS];
  int64_t ld;                 // elements between rows of W
  PoolDev pa, pb;
  const int64_t *a_start, *a_len;
  int adapter, n_slots_pool;
  int h_in, h_out;
  float scaling, sign;
  int n_ochunks;
  int chunks;                 // slices of merge_bm() input rows per workgroup
};

template <typename T, int KB>
__global__ __launch_bounds__(256, merge_resident(KB)) void merge_kernel(MergeArgs p) {
  using Tr = Traits<T>;
  using vec8 = typename Tr::vec8;
  constexpr int MG_BM = merge_bm(KB);
  constexpr int UNITS = KB * 4;      // 16-byte units (8 rank elements) per input row of the A slice
  __shared__ __align__(16) u32x4 s_a[MG_BM * UNITS];   // unit c of row i at b_swizzle(i * UNITS + c)
  __shared__ __align__(16) float stage[4][16][MG_STAGE_LD];   // (it also turns 16-byte units)

  const int z = blockIdx.y;
  const int slot = p.slots[z];
  uint16_t *__restrict__ W = p.w[z];
  const int itile = blockIdx.x / p.n_ochunks;
  const int oc = blockIdx.x - itile * p.n_ochunks;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 15, kg = lane >> 4;
  const int o_wave = oc * MG_BN + wave * 64;

  // ranks are at most 128, so a usable length fits 32 bits (a 64-bit division would cost the set-up some 0.2 us)
  const int64_t alen = p.a_len[p.adapter];
  const int r = alen > 0 && alen < (1 << 20) ? (int)((uint32_t)alen / (uint32_t)p.n_slots_pool) : 0;
  if (r <= 0 || (r & 7) || r > KB * 32) return;      // same adapters the LoRA op accepts
  const int64_t base = p.a_start[p.adapter] + (int64_t)r * slot;

  // Row-major roles for the update of W: 8 lanes x 16 bytes cover one row of the wave's 64 outputs.
  const int rr0 = lane >> 3, c8 = (lane & 7) * 8;
  const bool ocol_ok = (o_wave + c8) < p.h_out;

  const float inv_h_out = 1.0f / (float)p.h_out;
  // ---- a thread's 8 x 8 block of an A slice: rank rows 8 * ac .. + 8, 16 bytes of input columns from 8 * aic on.
  // Neighbouring threads take neighbouring chunks of the same rank rows: whole lines.  The first slice's block is
  // requested before anything waits for B where the registers are there: above rank 64, with two workgroups resident.
  // (Below, with four, it spills: at ranks up to 32 without it 3072 wide 273 -> 270 us, 4096 wide 409 -> 405 for eight
  // calls of four slots.)
  constexpr int CHUNKS = MG_BM / 8;
  static_assert(CHUNKS * UNITS <= 256, "one block per thread");
  const int ac = tid / CHUNKS, aic = tid - ac * CHUNKS;
  const int row0 = itile * p.chunks * MG_BM;
  const int n_rows = min(p.chunks * MG_BM, p.h_in - row0);        // of this workgroup
  // All look-ups in one round trip: those with nothing to look up read entry 0 (the host has checked that there is one).
  int64_t alook[8], blook[KB][4];
  uint32_t boff[KB][4];
  bool aok[8], bok[KB][4];
#pragma unroll
  for (int jj = 0; jj < 8; ++jj) {
    const int64_t ai = base + ac * 8 + jj;
    aok[jj] = ac * 8 + jj < r && ai >= 0 && ai < p.pa.a_loc_len;
    alook[jj] = p.pa.a_loc[aok[jj] ? ai : 0];
  }
#pragma unroll
  for (int q = 0; q < KB; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t flat, bin;
      bok[q][i] = b_unit<KB>(q, i, lane, (uint32_t)r, (uint32_t)o_wave * (uint32_t)r, flat);   // < 2^16 * 2^7
      divmod24(flat, (uint32_t)p.h_out, inv_h_out, bin, boff[q][i]);
      const int64_t idx = base + bin;
      bok[q][i] = bok[q][i] && flat < (uint32_t)p.h_out * (uint32_t)r && idx >= 0 && idx < p.pb.a_loc_len;
      blook[q][i] = p.pb.a_loc[bok[q][i] ? idx : 0];
    }
  int arow[8];
#pragma unroll
  for (int jj = 0; jj < 8; ++jj)   // pool rows fit 31 bits (checked on the host)
    arow[jj] = aok[jj] && alook[jj] >= 0 && alook[jj] < p.pa.w_rows ? (int)alook[jj] : -1;
  u32x4 ablk[8];
  auto load_a = [&](int il0) {
    const int il = il0 + aic * 8;
#pragma unroll
    for (int jj = 0; jj < 8; ++jj)
      ablk[jj] = (arow[jj] >= 0 && il < n_rows) ? load16(p.pa.w + (int64_t)arow[jj] * p.h_in + row0 + il)
                                                : u32x4{0, 0, 0, 0};
  };
  // ---- B units, then B fragments, scaled and rounded to T: bfrag[nb][kb] = T(B^T[o][j0..j0+8) * scaling)
  u32x4 braw[KB][4], bfrag[4][KB];
#pragma unroll
  for (int q = 0; q < KB; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool ok = bok[q][i] && blook[q][i] >= 0 && blook[q][i] < p.pb.w_rows;
      braw[q][i] = ok ? load16(p.pb.w + blook[q][i] * p.h_out + boff[q][i]) : u32x4{0, 0, 0, 0};
    }
  constexpr bool A_FIRST = merge_resident(KB) <= 2;
  if constexpr (A_FIRST) load_a(0);
  static_assert(sizeof(stage) / 4 >= B_TURN_BYTES, "a wave's staging tile holds its turn");
  b_turn<KB>(braw, bfrag, (uint32_t)r, r, lane, reinterpret_cast<unsigned char *>(&stage[wave][0][0]));
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      float f[8];
      unpack8<T>(bfrag[nb][kb], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        // the reference's `B * scaling` is an fp32 product rounded to T afterwards: keep the two roundings
        // apart (a fused multiply-and-convert rounds once and differs whenever the fp32 product lands on a
        // tie of T, which decimal scalings such as 1.7 or 0.9 do for a few percent of the elements)
        f[e] *= p.scaling;
        asm volatile("" : "+v"(f[e]));
      }
      bfrag[nb][kb] = pack8<T>(f);
    }

  uint16_t *const wbase = W + (int64_t)row0 * p.ld + o_wave + c8;
  u32x4 wv[2][2];
  auto load_w = [&](int il0) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int il = il0 + b * 16 + rr0 + 8 * h;
        wv[b][h] = (ocol_ok && il < n_rows) ? load16(wbase + (int64_t)il * p.ld) : u32x4{0, 0, 0, 0};
      }
  };
#pragma unroll 1
  for (int ch = 0; ch * MG_BM < n_rows; ++ch) {
    // ---- the [r x MG_BM] slice of A into LDS, transposed (rank rows beyond r are zero); the swizzle spreads the
    // units of neighbouring threads over the banks
    if (ch > 0 || !A_FIRST) load_a(ch * MG_BM);
    if (ch > 0) __syncthreads();   // everybody has read the previous slice
    if (tid < CHUNKS * UNITS) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        u32x4 unit;
#pragma unroll
        for (int w = 0; w < 4; ++w)   // element e of rank rows 2w and 2w + 1
          unit[w] = __builtin_amdgcn_perm(ablk[2 * w + 1][e >> 1], ablk[2 * w][e >> 1], (e & 1) ? 0x07060302u : 0x05040100u);
        s_a[b_swizzle((uint32_t)((aic * 8 + e) * UNITS + ac))] = unit;
      }
    }
    __syncthreads();

#pragma unroll 1
    for (int rb0 = 0; rb0 < MG_BM / 16; rb0 += 2) {
      load_w(ch * MG_BM + rb0 * 16);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        // A^T fragment: row = input row (lrow), 8 consecutive rank elements
        u32x4 afrag[KB];
        const int al = (rb0 + b) * 16 + lrow;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) afrag[kb] = s_a[b_swizzle((uint32_t)(al * UNITS + kb * 4 + kg))];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
            if (kb * 32 < r) acc = Tr::mfma(as<vec8>(afrag[kb]), as<vec8>(bfrag[nb][kb]), acc);
#pragma unroll
          for (int t = 0; t < 4; ++t) stage[wave][kg * 4 + t][nb * 16 + lrow] = acc[t];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int il = ch * MG_BM + (rb0 + b) * 16 + rr0 + 8 * h;
          if (ocol_ok && il < n_rows) {
            const float *srow = &stage[wave][rr0 + 8 * h][c8];
            float f[8];
            unpack8<T>(wv[b][h], f);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              const float ab = Tr::to_float(Tr::from_float(srow[k]));   // the GEMM result is a T tensor
              f[k] += p.sign * ab;
            }
            store16(wbase + (int64_t)il * p.ld, pack8<T>(f));
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
}

template <typename T>
int launch_merge_t(hipStream_t st, const MergeArgs &a, int kb, dim3 grid) {
  switch (kb) {
    case 1: hipLaunchKernelGGL((merge_kernel<T, 1>), grid, dim3(256), 0, st, a); break;
    case 2: hipLaunchKernelGGL((merge_kernel<T, 2>), grid, dim3(256), 0, st, a); break;
    case 4: hipLaunchKernelGGL((merge_kernel<T, 4>), grid, dim3(256), 0, st, a); break;
    default: return fail(MLORA_ERR_NO_KERNEL, "merge: no kernel for %d rank blocks", kb);
  }
  return check_launch("merge_kernel");
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

}  // namespace mlora

using namespace mlora;

extern "C" int mlora_merge_adapter(void *stream, void *const *w, const int32_t *slots, int32_t n_targets, int64_t ld,
                                   int64_t h_in, int64_t h_out, const mlora_pool *pool_a, const mlora_pool *pool_b,
                                   int64_t adapter, int64_t max_rank, float scaling, int32_t sign, mlora_dtype dtype) {
  if (dtype != MLORA_F16 && dtype != MLORA_BF16)
    return fail(MLORA_ERR_NO_KERNEL, "No suitable kernel. h_in=%lld h_out=%lld dtype=%d", (long long)h_in,
                (long long)h_out, (int)dtype);
  if (!pool_a || !pool_b || !w || !slots) return fail(MLORA_ERR_INVALID, "merge_adapter: null pointer");
  if (n_targets < 1 || n_targets > MLORA_MAX_TARGETS)
    return fail(MLORA_ERR_INVALID, "merge_adapter: n_targets=%d outside [1,%d]", n_targets, MLORA_MAX_TARGETS);
  if (h_in <= 0 || h_out <= 0 || h_in >= 65536 || h_out >= 65536 || (h_in % 8) || (h_out % 8) || ld < h_out || (ld % 8))
    return fail(MLORA_ERR_NO_KERNEL, "No suitable kernel. h_in=%lld h_out=%lld ld=%lld", (long long)h_in,
                (long long)h_out, (long long)ld);
  if (max_rank <= 0 || max_rank > MAX_RANK || (max_rank % 8))
    return fail(MLORA_ERR_NO_KERNEL, "merge_adapter: max_rank=%lld not a multiple of 8 in (0,%d]", (long long)max_rank,
                MAX_RANK);
  if (adapter < 0 || adapter >= pool_a->n_adapters || pool_a->n_adapters != pool_b->n_adapters)
    return fail(MLORA_ERR_INVALID, "merge_adapter: adapter %lld outside [0,%lld)", (long long)adapter,
                (long long)pool_a->n_adapters);
  // (the kernel keeps pool rows in 31 bits)
  if (pool_a->a_loc_len > 0x7fffffff || pool_a->w_rows > 0x7fffffff || pool_b->a_loc_len > 0x7fffffff || pool_b->w_rows > 0x7fffffff)
    return fail(MLORA_ERR_NO_KERNEL, "merge_adapter: more than 2^31 - 1 index entries or pool rows");
  if (sign != 1 && sign != -1) return fail(MLORA_ERR_INVALID, "merge_adapter: sign must be +1 or -1");
  if (!pool_a->w || !pool_b->w || !pool_a->a_start || !pool_a->a_len || !pool_a->a_loc || !aligned16(pool_a->w) ||
      !aligned16(pool_b->w))
    return fail(MLORA_ERR_INVALID, "merge_adapter: pool tensors are null or misaligned");
  MergeArgs a;
  for (int i = 0; i < MLORA_MAX_TARGETS; ++i) {
    const int k = i < n_targets ? i : 0;
    if (!w[k] || !aligned16(w[k])) return fail(MLORA_ERR_INVALID, "merge_adapter: weight %d is null or misaligned", k);
    if (slots[k] < 0 || slots[k] >= pool_a->n_slots)
      return fail(MLORA_ERR_INVALID, "merge_adapter: slot %d outside [0,%d)", slots[k], pool_a->n_slots);
    a.w[i] = static_cast<uint16_t *>(w[k]);
    a.slots[i] = slots[k];
  }
  if (pool_a->a_loc_len < 1 || pool_b->a_loc_len < 1) return MLORA_OK;  // no rows to merge; the kernel reads entry 0
  a.ld = ld;
  a.pa = PoolDev{static_cast<const uint16_t *>(pool_a->w), pool_a->w_rows, pool_a->a_loc, pool_a->a_loc_len};
  a.pb = PoolDev{static_cast<const uint16_t *>(pool_b->w), pool_b->w_rows, pool_b->a_loc, pool_b->a_loc_len};
  a.a_start = pool_a->a_start;
  a.a_len = pool_a->a_len;
  a.adapter = (int)adapter;
  a.n_slots_pool = pool_a->n_slots;
  a.h_in = (int)h_in;
  a.h_out = (int)h_out;
  a.scaling = scaling;
  a.sign = (float)sign;
  a.n_ochunks = (int)((h_out + MG_BN - 1) / MG_BN);
  int kb = (int)((max_rank + 31) / 32);
  kb = kb <= 1 ? 1 : kb <= 2 ? 2 : 4;
  const int bm = merge_bm(kb);
  // Slices per workgroup.  The grid takes so many rounds of what the device holds, each as long as a workgroup's slices
  // and its set-up, which with the B fragments of rank 64 and more costs about one slice more (rank 128, 4096 wide: one
  // slice 85.6 us, two 73.6, four 68.8; 3072 wide: 59.8, 62.8, three 51.1, four 59.1; rank 64, 4096 wide: 66.3, two 59.0,
  // four 64.0).  Up to rank 32 one slice is always fastest (rank 16, 4096 wide: 56.5, two 59.8).
  const int64_t slices = (h_in + bm - 1) / bm, per_slice = (int64_t)a.n_ochunks * n_targets;
  const int64_t resident = (int64_t)merge_resident(kb) * 256;
  auto cost = [&](int64_t c) { return ((slices + c - 1) / c * per_slice + resident - 1) / resident * (c + 1); };
  a.chunks = 1;
  for (int c = 2; kb > 1 && c <= 4; ++c)
    if (cost(c) < cost(a.chunks)) a.chunks = c;
  const int64_t blocks = (slices + a.chunks - 1) / a.chunks * a.n_ochunks;
  dim3 grid((unsigned)blocks, (unsigned)n_targets);
  return dtype == MLORA_F16 ? launch_merge_t<_Float16>((hipStream_t)stream, a, kb, grid)
                            : launch_merge_t<__bf16>((hipStream_t)stream, a, kb, grid);
}
