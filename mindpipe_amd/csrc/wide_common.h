// Device helpers of the direct-to-LDS GEMMs (dqwide.hip, i8wide.hip, w4wide.hip).
#pragma once
#include "mp_common.h"

namespace {

typedef __bf16 wbf8_t __attribute__((ext_vector_type(8)));
typedef __bf16 wbf2_t __attribute__((ext_vector_type(2)));
typedef _Float16 whf2_t __attribute__((ext_vector_type(2)));

constexpr int kWBK = 64;                 // K step
constexpr int kWLds = 160 * 1024;         // one workgroup per CU
constexpr int kWLgkm0 = 0xC07F;          // s_waitcnt lgkmcnt(0)
constexpr uint32_t kWOob = 0x80000000u;  // past every descriptor: zeros, no memory access

// In a non-template function: with an operand that depends on a template parameter the cast to an LDS
// pointer makes the host pass drop the kernel's launch stub.
__device__ __forceinline__ void wide_lds_load16(__amdgpu_buffer_rsrc_t r, int8_t *lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, reinterpret_cast<__attribute__((address_space(3))) void *>(reinterpret_cast<uintptr_t>(lds)), 16, voff,
      __builtin_amdgcn_readfirstlane(static_cast<int>(soff)), 0, 0);
}

// The end of a phase of the K loop: nothing moves across it, in either direction.
__device__ __forceinline__ void wide_phase() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Whether wide_tile deals the row slots of the last column tiles (see there).
__host__ __device__ __forceinline__ bool wide_by_slot(const void *offsets, int n_experts, int64_t slots) {
  return offsets != nullptr && n_experts > 1 && slots >= 8;
}

// Column tile, row slot and K split of a workgroup, of `cols` x `slots` x `splits`; false if it has none.  Workgroups go to
// the eight XCDs by turns; the row slots and splits of a column tile stay on one XCD, whose L2 then serves what they
// share, and column tiles are dealt to the XCDs, but for the last cols % 8: those are cut into eight equal runs.
// (Dealt as well, they left 20 tiles a third short of work on half of the XCDs and 4 tiles half of the XCDs idle:
// M = 3072, 5120 x 5120 in int8 126 -> 77 us, M = 12288, N = 1024, K = 4096 106 -> 56 us.)  With several groups (splits = 1)
// the last slots of a column are often empty and runs are not equal work: from a slot per XCD, the slots of the last
// columns are dealt (64 experts, 192 rows each, gate / up of 512 x 2048 with the requantization: 94 ->
// 61 us).
__device__ __forceinline__ bool wide_tile(int bx, int cols, int slots, int splits, bool by_slot, int &col, int &slot, int &sp) {
  const int x = bx & 7, per = slots * splits, whole = cols / 8 * per, last = cols % 8, tail = last * per;
  int j = bx >> 3;
  if (by_slot && j >= whole) {
    j -= whole;
    const int n = last > 0 ? last : 1;
    slot = __builtin_amdgcn_readfirstlane(j / n * 8 + x);
    col = __builtin_amdgcn_readfirstlane(cols / 8 * 8 + j % n);
    sp = 0;
    return last > 0 && slot < slots;
  }
  const bool dealt = j < whole;
  j -= dealt ? 0 : whole;
  const bool ok = dealt || j < tail / 8 + (x < tail % 8 ? 1 : 0);
  j += dealt ? 0 : x * (tail / 8) + min(x, tail % 8);
  col = __builtin_amdgcn_readfirstlane(dealt ? j / per * 8 + x : cols / 8 * 8 + j / per);
  slot = __builtin_amdgcn_readfirstlane(j % per / splits);
  sp = __builtin_amdgcn_readfirstlane(j % per % splits);
  return ok;
}

// Rows [rb, re) and expert of row slot `slot` (dense: the slot-th 256 of `rows`; grouped: the slot-th 256-row chunk of an
// expert, in expert order); false past the last one.  Called by whole waves; the results are uniform.  Each lane
// looks at one expert and a prefix sum finds the slot's: taken one after the other, the loads of a search through
// 256 experts held each workgroup up for about 13 us.
__device__ __forceinline__ bool wide_rows(const int64_t *offsets, int n_experts, int64_t rows, int slot, int64_t &rb,
                                          int64_t &re, int &expert) {
  expert = 0;
  if (!offsets) {
    rb = static_cast<int64_t>(slot) * 256;
    re = rb + 256 < rows ? rb + 256 : rows;
    return rb < rows;
  }
  const int lane = threadIdx.x & 63;
  for (int e0 = 0; e0 < n_experts; e0 += 64) {
    const int e = min(e0 + lane, n_experts - 1);
    const int lo = static_cast<int>(offsets[e]), hi = static_cast<int>(offsets[e + 1]);
    const int nch = e0 + lane < n_experts && hi > lo ? (hi - lo + 255) / 256 : 0;
    int upto = nch;  // chunks of the experts up to this lane's
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, 64);
      upto += lane >= o ? v : 0;
    }
    const uint64_t past = __ballot(upto > slot);
    if (past) {
      const int l = __builtin_ctzll(past);
      const int first = __builtin_amdgcn_readlane(lo, l), end = __builtin_amdgcn_readlane(hi, l);
      rb = first + (slot - __builtin_amdgcn_readlane(upto - nch, l)) * 256;
      re = rb + 256 < end ? rb + 256 : end;
      expert = e0 + l;
      return true;
    }
    slot -= __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

template <int DT>
__device__ __forceinline__ uint32_t wide_pack2(float a, float b) {
  if constexpr (DT == MP_F16) {
    const whf2_t v = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
    return __builtin_bit_cast(uint32_t, v);
  } else {
    const wbf2_t v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
    return __builtin_bit_cast(uint32_t, v);
  }
}

template <int DT>
__device__ __forceinline__ f16_t wide_mfma(i4_t a, uint4 b, f16_t c) {
  if constexpr (DT == MP_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8_t, a), __builtin_bit_cast(h8_t, b), c, 0, 0,
                                                  0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(wbf8_t, a), __builtin_bit_cast(wbf8_t, b), c, 0,
                                                   0, 0);
}

template <int N>
__device__ __forceinline__ void wide_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One 32 x 32 fp32 MFMA tile of a K split to the partials, through a wave-private LDS tile of 144-byte rows:
// accumulator r is row 8 (r >> 2) + 4 half + (r & 3), column lane % 32; a lane then stores four columns of a row.
// `rows` and `cols` bound what is stored of the tile, `ld` is the row stride (elements), dst the tile's corner.
__device__ __forceinline__ void wide_store_part(const f16_t &acc, int8_t *stage, float *dst, int64_t ld, int rows, int cols,
                                                int lane) {
#pragma unroll
  for (int r = 0; r < 16; ++r)
    *reinterpret_cast<float *>(stage + (8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * 144 + (lane & 31) * 4) = acc[r];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = q * 8 + lane / 8, col = (lane & 7) * 4;
    const f4_t v = *reinterpret_cast<const f4_t *>(stage + row * 144 + (lane & 7) * 16);
    if (row >= rows) continue;
    float *d = dst + row * ld + col;
    if (ld % 4 == 0) {
      if (col < cols) *reinterpret_cast<f4_t *>(d) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < cols) d[e] = v[e];
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the next tile overwrites the region
}

// Sums of the K splits' fp32 partials [splits, m, n] in split order, plus bias, rounded once; four columns per thread.
template <int DT>
__global__ __launch_bounds__(256) void wide_reduce_kernel(const float *__restrict__ part, int splits, int64_t m, int64_t n,
                                                          const uint16_t *__restrict__ bias, uint16_t *__restrict__ y) {
  const int64_t per = (n + 3) / 4, t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= m * per) return;
  const int64_t row = t / per, c = t % per * 4;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < splits; ++s) {
    const float *src = part + (s * m + row) * n + c;
    if (n % 4 == 0) {
      const float4 w = *reinterpret_cast<const float4 *>(src);
      v[0] = mp_add(v[0], w.x);
      v[1] = mp_add(v[1], w.y);
      v[2] = mp_add(v[2], w.z);
      v[3] = mp_add(v[3], w.w);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < n) v[e] = mp_add(v[e], src[e]);
    }
  }
  uint16_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float f = bias && c + e < n ? mp_add(v[e], mp_load_as_f32(bias, c + e, DT)) : v[e];
    o[e] = DT == MP_F16 ? mp_f2h(f) : mp_f2bf(f);
  }
  uint16_t *d = y + row * n + c;
  if (n % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0) {
    *reinterpret_cast<uint2 *>(d) = make_uint2(o[0] | (static_cast<uint32_t>(o[1]) << 16), o[2] | (static_cast<uint32_t>(o[3]) << 16));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < n) d[e] = o[e];
  }
}

// Ways to split K over workgroups so that tiles of 256 rows x 128 columns give each CU one: at least K = 1024
// each, at most 8.
inline int wide_splits(int64_t m, int64_t n, int64_t k) {
  const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256;
  const int64_t tiles = mp_cdiv(n, 128) * mp_cdiv(m, 256);
  int64_t s = cus / tiles;
  if (s > k / 1024) s = k / 1024;
  if (s > 8) s = 8;
  return s < 1 ? 1 : static_cast<int>(s);
}

template <int DT>
int wide_reduce(const float *part, int splits, int64_t m, int64_t n, const void *bias, void *y, hipStream_t stream) {
  hipLaunchKernelGGL((wide_reduce_kernel<DT>), dim3(static_cast<unsigned>(mp_cdiv(m * mp_cdiv(n, 4), 256))), dim3(256), 0,
                     stream, part, splits, m, n, static_cast<const uint16_t *>(bias), static_cast<uint16_t *>(y));
  MP_CHECK_LAUNCH();
  return MP_OK;
}

}  // namespace

// Row slots of 256 that hold any split of `rows` into `groups` groups: sum ceil(r / 256) <= (rows + 255 groups) / 256.
// No more than that: workgroups go to the shader engines by turns, and a single group's spare slot (every other
// workgroup empty) left half of the engines idle (200 rows, 11008 gate / up pairs x 4096: 74 -> 43 us).
static inline int64_t wide_row_slots(int64_t rows, int64_t groups) {
  return (rows + 255 * (groups < rows ? groups : rows)) / 256;
}

// Workgroups of wide_tile's dealing: as many for each XCD as the one with the most has.
static inline int64_t wide_grid(int64_t cols, int64_t slots, int64_t splits, bool by_slot) {
  const int64_t tail = by_slot ? mp_cdiv(slots, 8) * (cols % 8) : mp_cdiv(cols % 8 * slots * splits, 8);
  return 8 * (cols / 8 * slots * splits + tail);
}
