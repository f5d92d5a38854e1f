// The direct-to-LDS int8 GEMM, a workgroup up to 256 rows of one weight, dense (any number of row slots) or grouped by
// expert: the phases, the wave roles and the stages of dq_wide_kernel (dqwide.hip) on int8 operands and the int8 matrix
// cores.
//
// What bounds it: the weight stream (a decode batch or a few hundred rows per expert); with thousands of rows the int8
// rate that the card's power allows (M = 4096, N = 11008, K = 4096 1.8 POP/s traced, a library product of 8192^3 2.16).
// Register staging keeps two K steps in flight per CU; here the rest of the 160 KB of LDS is weight stages, the loads go
// out between MFMAs, and the XCDs start at different places of K so that the workgroups do not all ask for the same
// bytes of rows that lie K apart.
#include "i8_wide.h"
#include "wide_common.h"

#include <type_traits>

namespace {

constexpr int kI8BK = 128;

// A workgroup of eight waves (two along M, four along N): up to 256 rows x BN = 128 TN weight rows (SwiGLU: BN / 2
// gate rows and the BN / 2 matching up rows), a wave up to 4 x TN MFMA 32x32x32 tiles, row tiles 2 i + wm.  LDS:
// three activation stages of K = 128 sized by the row tiles that are there, weight stages of K = 128 in the rest;
// 128-byte rows, 16-byte chunk c of row r at slot c ^ ((r >> 1) & 7).  Waves 0..3 load the weights, 4..7 the
// activations, and run one phase apart.  SwiGLU with TN = 1: a wave's 32 weight rows are 16 gate rows and their up
// rows.  PART: split `part` of the K steps, int32 sums to p.y [splits, rows, n].
template <int EPI, int TN, bool PART>
__global__ __launch_bounds__(512, 2) void i8_wide_kernel(mp_i8_args p, int n_slots, int splits) {
  constexpr bool SWI = EPI == MP_EPI_SWIGLU;
  constexpr int TM = 4, WN = 4, BN = 128 * TN;
  constexpr int QB = BN / 8 / 4;
  constexpr int BST = BN * 128;
  static_assert(!(SWI && PART), "forms");
  extern __shared__ __attribute__((aligned(16))) int8_t smem_i8w[];
  const int bx = static_cast<int>(blockIdx.x);
  constexpr int CPT = SWI ? BN / 2 : BN;  // output columns of a tile
  int col, slot, part;
  if (!wide_tile(bx, static_cast<int>((p.n + CPT - 1) / CPT), n_slots, PART ? splits : 1,
                 wide_by_slot(p.offsets, p.n_experts, n_slots), col, slot, part))
    return;
  int64_t rb, re;
  int expert;
  if (!wide_rows(p.offsets, p.n_experts, p.rows, slot, rb, re, expert)) return;  // workgroup-uniform
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, half = lane >> 5;
  const uint32_t k = static_cast<uint32_t>(p.k);
  const int rows = static_cast<int>(re - rb);
  const int n_out = static_cast<int>(p.n), c0 = col * CPT;
  const int64_t nb_rows = SWI ? 2 * p.n : p.n;
  const int nt = (rows + 31) / 32;
  const int nv = nt > wm ? (nt - wm + 1) / 2 : 0;
  const int ast = nt * 32 * 128, b0 = 3 * ast;
  const int nbs = min(6, (kWLds - (nt & 1) * 1024 - b0) / BST);

  const auto arsrc = mp_rsrc(p.a + rb * p.k, static_cast<uint32_t>(rows) * k);
  const auto brsrc = mp_rsrc(p.b + expert * nb_rows * p.k, static_cast<uint32_t>(nb_rows) * k);
  uint32_t voff[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = (q * 4 + wn) * 8 + lane / 8;
    const uint32_t ch = 16 * ((lane & 7) ^ ((r >> 1) & 7));
    if (wm == 1) {
      voff[q] = r < rows ? static_cast<uint32_t>(r) * k + ch : kWOob;
    } else {
      // SwiGLU: BN / 2 gate rows then their up rows, with one tile per wave 16 gate and 16 up rows by turns
      const int c = c0 + (!SWI ? r : (TN == 2 ? r % (BN / 2) : r / 32 * 16 + r % 16));
      const bool up = SWI && (TN == 2 ? r >= BN / 2 : r % 32 >= 16);
      const uint32_t row = static_cast<uint32_t>(c + (up ? n_out : 0));
      voff[q] = c < n_out && r < BN ? row * k + ch : kWOob;
    }
  }
  const int steps = static_cast<int>(k / kI8BK);
  const int first = PART ? steps * part / splits : 0, nkt = (PART ? steps * (part + 1) / splits : steps) - first;
  const int rot = ((bx & 7) * nkt / 8 + expert * 5) % nkt;
  auto at = [&](int t) {  // byte offset of step t of the range; past its end a step again, never read
    t += rot;
    return (first + min(t < nkt ? t : t - nkt, nkt - 1)) * kI8BK;
  };
  auto load_a = [&](int kt, int slot, int q) {
    const int g = q * 4 + wn;
    wide_lds_load16(arsrc, smem_i8w + (g < nt * 4 ? slot * ast + g * 1024 : kWLds - 1024), voff[q], at(kt));
  };
  auto load_b = [&](int kt, int slot, int q) {
    wide_lds_load16(brsrc, smem_i8w + b0 + slot * BST + (q * 4 + wn) * 1024, voff[q], at(kt));
  };
  auto wait_b = [&](int n) {  // at most n weight stages still in flight
    if (n <= 0) wide_wait_vm<0>();
    else if (n == 1) wide_wait_vm<QB>();
    else if (n == 2) wide_wait_vm<2 * QB>();
    else if (n == 3) wide_wait_vm<3 * QB>();
    else wide_wait_vm<4 * QB>();
  };

  i16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
  const int swz = (lane >> 1) & 7;
  const int abase = (wm * 32 + (lane & 31)) * 128;
  const int bbase = b0 + ((SWI ? wn * 32 : wn * TN * 32) + (lane & 31)) * 128;

  auto k_loop = [&](auto h_, auto nv_, auto wm_) {
    constexpr int H = decltype(h_)::value, NV = decltype(nv_)::value, WMC = decltype(wm_)::value;
    constexpr int NC = H * TN > 6 ? 2 : 4;       // MFMA operands (K = 32) per phase
    constexpr int NM = NC * NV * TN;             // MFMAs of a phase
    constexpr int QL = WMC == 1 ? 2 * H : QB;    // loads of a step
    if constexpr (WMC == 1) {
#pragma unroll
      for (int st = 0; st < 3; ++st)
#pragma unroll
        for (int q = 0; q < 2 * H; ++q) load_a(st, st, q);
      wide_wait_vm<4 * H>();
    } else {
      for (int st = 0; st < nbs - 1; ++st)
#pragma unroll
        for (int q = 0; q < QB; ++q) load_b(st, st, q);
      wait_b(nbs - 2);
    }
    wide_phase();
    if constexpr (WMC == 1) wide_phase();
    __builtin_amdgcn_s_waitcnt(kWLgkm0);  // only LDS reads are counted inside the loop
    int sa = 0, sb = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      const int8_t *pa = smem_i8w + sa * ast, *pb = smem_i8w + sb * BST;
#pragma unroll
      for (int k0 = 0; k0 < 4; k0 += NC) {
        i4_t bf[NC][TN], af[NC][NV > 0 ? NV : 1];
        if constexpr (NV > 0) {
#pragma unroll
          for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
              bf[c][j] = *reinterpret_cast<const i4_t *>(pb + bbase + j * (SWI ? BN / 2 : 32) * 128 +
                                                         16 * ((2 * (k0 + c) + half) ^ swz));
#pragma unroll
            for (int i = 0; i < NV; ++i)
              af[c][i] = *reinterpret_cast<const i4_t *>(pa + abase + i * 2 * 32 * 128 +
                                                         16 * ((2 * (k0 + c) + half) ^ swz));
          }
        }
        if (WMC == 1 && k0 + NC == 4) wide_wait_vm<2 * H>();  // the next step's activations have landed
        __builtin_amdgcn_s_waitcnt(kWLgkm0);
        wide_phase();
        __builtin_amdgcn_s_setprio(1);
        // loads into stages that every wave has read: the activations three steps on, the last weight stage
        const bool loads = WMC == 1 ? k0 + NC == 4 : k0 == 0;
        auto load = [&](int q) {
          if (WMC == 1) load_a(kt + 3, sa, q);
          else load_b(kt + nbs - 1, sb == 0 ? nbs - 1 : sb - 1, q);
        };
        if constexpr (NV > 0) {
#pragma unroll
          for (int x = 0; x < NM; ++x) {
            const int c = x / (NV * TN), i = x / TN % NV, j = x % TN;
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[c][i], bf[c][j], acc[i][j], 0, 0, 0);
            if (loads) {
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int q = x * QL / NM; q < (x + 1) * QL / NM; ++q) load(q);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        } else if (loads) {
#pragma unroll
          for (int q = 0; q < QL; ++q) load(q);
        }
        __builtin_amdgcn_s_setprio(0);
        if (WMC == 0 && k0 + NC == 4) wait_b(nbs - 2);  // the next step's weights have landed
        wide_phase();
      }
      sa = sa == 2 ? 0 : sa + 1;
      sb = sb == nbs - 1 ? 0 : sb + 1;
    }
    if constexpr (WMC == 0) wide_phase();
  };
  auto by_rows = [&](auto h_) {
    constexpr int H = decltype(h_)::value;
    if (wm == 0) k_loop(h_, h_, std::integral_constant<int, 0>{});
    else if (nv == H) k_loop(h_, h_, std::integral_constant<int, 1>{});
    else k_loop(h_, std::integral_constant<int, H - 1>{}, std::integral_constant<int, 1>{});
  };
  if (nt > 6) by_rows(std::integral_constant<int, 4>{});
  else if (nt > 4) by_rows(std::integral_constant<int, 3>{});
  else if (nt > 2) by_rows(std::integral_constant<int, 2>{});
  else by_rows(std::integral_constant<int, 1>{});
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // no LDS load in flight, every stage read

  // ---- epilogue, one 32 x 32 tile at a time through a wave-private LDS tile of 32-bit values (row stride 144 bytes):
  // accumulator r is row 8 (r >> 2) + 4 half + (r & 3), column lane % 32; a lane then holds four columns of a row
  constexpr int LDR = 144;
  int8_t *stage = smem_i8w + wave * (32 * LDR);
  float *stok = reinterpret_cast<float *>(smem_i8w + 8 * 32 * LDR);  // per-token scales of the 256 rows
  if (!PART) {
    if (tid < 256) stok[tid] = tid < rows ? p.s_a[rb + tid] : 0.f;
    mp_lds_barrier();
  }
  const float *sbx = p.s_b + expert * nb_rows;
  char *yb = static_cast<char *>(p.y);
  const int esz = PART || SWI || EPI == MP_EPI_F32 || p.out_dtype == MP_F32 ? 4 : 2;
  const bool vec = n_out % 4 == 0 && p.ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(p.y) & (4 * esz - 1)) == 0;
  const int64_t prow = PART ? part * p.rows : 0;
  if constexpr (SWI && TN == 1) {
    // a wave's tile is 16 gate columns and the matching 16 up columns: the products meet in the staged tile, a lane
    // then holds two output columns of a row; the abs-max of 32 columns joins two waves' in LDS
    float *samax = stok + 256;  // [256 rows][4 wave columns]
    const int cw0 = c0 + wn * 16, cl = min(cw0 + (lane & 15), n_out - 1);
    const float sc = sbx[((lane & 16) ? n_out : 0) + cl];
    const bool pair = n_out % 2 == 0 && p.ldy % 2 == 0 && (reinterpret_cast<uintptr_t>(p.y) & 7) == 0;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (i >= nv) continue;  // wave-uniform
      const int lr = (i * 2 + wm) * 32;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f4_t st4 = *reinterpret_cast<const f4_t *>(stok + lr + 8 * g + 4 * half);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float *>(stage + (8 * g + 4 * half + e) * LDR + (lane & 31) * 4) =
              mp_mul(mp_mul(static_cast<float>(acc[i][0][4 * g + e]), st4[e]), sc);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = q * 8 + lane / 8, col = cw0 + (lane & 7) * 2;
        const int64_t m = rb + lr + row, o = m * p.ldy + col;
        float a = 0.f, h[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float *gu = reinterpret_cast<const float *>(stage + row * LDR) + (lane & 7) * 2 + e;
          h[e] = mp_swiglu_epi(gu[0], gu[16], p.epi_round);
          if (col + e < n_out) a = fmaxf(a, fabsf(h[e]));
        }
        a = fmaxf(a, __shfl_xor(a, 1, 64));
        a = fmaxf(a, __shfl_xor(a, 2, 64));
        a = fmaxf(a, __shfl_xor(a, 4, 64));
        if ((lane & 7) == 0) samax[(lr + row) * 4 + wn] = a;
        if (m >= re) continue;
        float *yo = reinterpret_cast<float *>(yb) + o;
        if (pair) {
          if (col < n_out) *reinterpret_cast<float2 *>(yo) = make_float2(h[0], h[1]);
        } else {
#pragma unroll
          for (int e = 0; e < 2; ++e)
            if (col + e < n_out) yo[e] = h[e];
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the next tile overwrites the region
    }
    mp_lds_barrier();
    const int row = tid / 2, w = (tid & 1) * 2;
    if (row < rows && c0 / 32 + (tid & 1) < p.n_partial)
      p.amax_partial[(rb + row) * p.n_partial + c0 / 32 + (tid & 1)] = fmaxf(samax[row * 4 + w], samax[row * 4 + w + 1]);
    return;
  }
  if constexpr (EPI == MP_EPI_DENSE && !PART) {
    // 16-bit outputs in whole 16-byte chunks: the wave's columns of a row tile staged as 16-bit values (row stride
    // 64 TN + 16 bytes), so that a row of the wave is one 64 TN byte segment of memory, in 16-byte stores (M = 4096,
    // 11008 x 4096 with the activations' quantization: 225 us through 32-bit tiles of 32 columns, 211 us)
    if (esz == 2 && n_out % 8 == 0 && p.ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0) {
      constexpr int CW = TN * 32, LD16 = CW * 2 + 16, CPR = CW / 8;  // 16-byte chunks per row
      const int cw0 = c0 + wn * CW;
      float sc[TN], bv[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int cl = min(cw0 + j * 32 + (lane & 31), n_out - 1);
        sc[j] = sbx[cl];
        bv[j] = p.bias != nullptr ? mp_load_as_f32(p.bias, cl, p.bias_dtype) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i >= nv) continue;  // wave-uniform
        const int lr = (i * 2 + wm) * 32;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f4_t st4 = *reinterpret_cast<const f4_t *>(stok + lr + 8 * g + 4 * half);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              float v = mp_mul(mp_mul(static_cast<float>(acc[i][j][4 * g + e]), st4[e]), sc[j]);
              if (p.bias != nullptr) v = mp_add(v, bv[j]);
              *reinterpret_cast<uint16_t *>(stage + (8 * g + 4 * half + e) * LD16 + (j * 32 + (lane & 31)) * 2) =
                  p.out_dtype == MP_F16 ? mp_f2h(v) : mp_f2bf(v);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int q = 0; q < CPR / 2; ++q) {
          const int row = (q * 64 + lane) / CPR, cc = (lane % CPR) * 8;
          const i4_t v = *reinterpret_cast<const i4_t *>(stage + row * LD16 + cc * 2);
          const int64_t m = rb + lr + row;
          if (m < re && cw0 + cc < n_out) *reinterpret_cast<i4_t *>(yb + (m * p.ldy + cw0 + cc) * 2) = v;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the next tile overwrites the region
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < (SWI ? 1 : TN); ++j) {
    const int cj = c0 + (SWI ? wn * 32 : (wn * TN + j) * 32);  // first column of the tile
    const int cl = cj + (lane & 31) < n_out ? cj + (lane & 31) : n_out - 1;
    const float sc = PART ? 0.f : sbx[cl], su = SWI ? sbx[n_out + cl] : 0.f;
    const bool hb = !PART && EPI == MP_EPI_DENSE && p.bias != nullptr;
    const float bv = hb ? mp_load_as_f32(p.bias, cl, p.bias_dtype) : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (i >= nv) continue;  // wave-uniform
      const int lr = (i * 2 + wm) * 32;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f4_t st4 = PART ? f4_t{} : *reinterpret_cast<const f4_t *>(stok + lr + 8 * g + 4 * half);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t o;
          if constexpr (PART) {
            o = static_cast<uint32_t>(acc[i][j][4 * g + e]);
          } else {
            float v = mp_mul(mp_mul(static_cast<float>(acc[i][j][4 * g + e]), st4[e]), sc);
            if constexpr (SWI)
              v = mp_swiglu_epi(v, mp_mul(mp_mul(static_cast<float>(acc[i][TN - 1][4 * g + e]), st4[e]), su), p.epi_round);
            else if (hb) v = mp_add(v, bv);
            o = __float_as_uint(v);
          }
          *reinterpret_cast<uint32_t *>(stage + (8 * g + 4 * half + e) * LDR + (lane & 31) * 4) = o;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = q * 8 + lane / 8, col = cj + (lane & 7) * 4;
        const i4_t v = *reinterpret_cast<const i4_t *>(stage + row * LDR + (lane & 7) * 16);
        const int64_t m = rb + lr + row;
        const bool ok = m < re;
        if constexpr (SWI) {
          float a = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < n_out) a = fmaxf(a, fabsf(__int_as_float(v[e])));
          a = fmaxf(a, __shfl_xor(a, 1, 64));
          a = fmaxf(a, __shfl_xor(a, 2, 64));
          a = fmaxf(a, __shfl_xor(a, 4, 64));
          if ((lane & 7) == 0 && ok && cj / 32 < p.n_partial) p.amax_partial[m * p.n_partial + cj / 32] = a;
        }
        if (!ok) continue;
        const int64_t o = (prow + m) * p.ldy + col;
        if (vec) {
          if (col >= n_out) continue;
          if (esz == 4) {
            *reinterpret_cast<i4_t *>(yb + o * 4) = v;
          } else {
            uint32_t h[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const float f0 = __int_as_float(v[2 * e]), f1 = __int_as_float(v[2 * e + 1]);
              h[e] = p.out_dtype == MP_F16 ? mp_f2h(f0) | (static_cast<uint32_t>(mp_f2h(f1)) << 16)
                                           : mp_f2bf(f0) | (static_cast<uint32_t>(mp_f2bf(f1)) << 16);
            }
            *reinterpret_cast<uint2 *>(yb + o * 2) = make_uint2(h[0], h[1]);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (col + e >= n_out) continue;
            if (esz == 4) reinterpret_cast<int *>(yb)[o + e] = v[e];
            else mp_store_from_f32(yb, o + e, p.out_dtype, __int_as_float(v[e]));
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the next tile overwrites the region
    }
  }
}

// Sums of the splits' int32 partials and the dense epilogue (acc * s_tok) * s_ch (+ bias), four columns per thread.
__global__ __launch_bounds__(256) void i8_reduce_kernel(const int *__restrict__ part, int splits, mp_i8_args p) {
  const int64_t per = (p.n + 3) / 4, t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= p.rows * per) return;
  const int64_t m = t / per, c = t % per * 4;
  const float st = p.s_a[m];
  int v[4] = {0, 0, 0, 0};
  const bool vec = p.n % 4 == 0;
  for (int s = 0; s < splits; ++s) {
    const int *src = part + (s * p.rows + m) * p.n + c;
    if (vec) {
      const int4 w = *reinterpret_cast<const int4 *>(src);
      v[0] += w.x;
      v[1] += w.y;
      v[2] += w.z;
      v[3] += w.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < p.n) v[e] += src[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (c + e >= p.n) break;
    float f = mp_mul(mp_mul(static_cast<float>(v[e]), st), p.s_b[c + e]);
    if (p.bias) f = mp_add(f, mp_load_as_f32(p.bias, c + e, p.bias_dtype));
    mp_store_from_f32(p.y, m * p.ldy + c + e, p.out_dtype, f);
  }
}

template <int EPI, int TN, bool PART>
int i8w_launch(const mp_i8_args &p, int splits, hipStream_t stream) {
  const int64_t slots = wide_row_slots(p.rows, p.offsets ? p.n_experts : 1);
  const int64_t wgs = wide_grid(mp_cdiv(p.n, EPI == MP_EPI_SWIGLU ? 64 * TN : 128 * TN), slots, splits,
                                wide_by_slot(p.offsets, p.n_experts, slots));
  if (wgs > INT32_MAX) return MP_ERR_SHAPE;
  const void *fn = reinterpret_cast<const void *>(i8_wide_kernel<EPI, TN, PART>);
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kWLds) != hipSuccess) return MP_ERR_HIP;
  hipLaunchKernelGGL((i8_wide_kernel<EPI, TN, PART>), dim3(static_cast<unsigned>(wgs)), dim3(512), kWLds,
                     stream, p, static_cast<int>(slots), splits);
  MP_CHECK_LAUNCH();
  return MP_OK;
}

}  // namespace

bool mp_i8_wide_takes(const mp_i8_args &p, int epi) {
  const int64_t nb_rows = epi == MP_EPI_SWIGLU ? 2 * p.n : p.n;
  return !p.shared_b && p.k % kI8BK == 0 && p.k <= (1 << 17) && nb_rows * p.k < (int64_t(1) << 31) && p.n < (1 << 28) &&
         p.rows > 0 && p.rows < (int64_t(1) << 31) && mp_aligned(p.a, 16) && mp_aligned(p.b, 16);
}

int mp_launch_i8_wide(const mp_i8_args &p, int epi, hipStream_t stream) {
  const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256;
  const int64_t groups = p.offsets ? (p.rows < p.n_experts ? p.rows : p.n_experts) : 1;
  const int64_t tiles = mp_cdiv(epi == MP_EPI_SWIGLU ? 2 * p.n : p.n, 256) * groups * mp_cdiv(mp_cdiv(p.rows, groups), 256);
  // 256 weight rows per workgroup: see wide_pick (dqwide.hip), and for a dense call also where tiles of 128 would be more
  // than one per CU, a second round of a few: M = 1280, 8192 x 8192 117 -> 103 us, M = 2304, N = 4096, K = 1024 27.7 ->
  // 22.8 us (23.1 on the large-M kernel); up to 128 rows, bound by the weight stream, 128 (M = 128, N = 40960, K = 8192 95
  // against 106 us)
  const bool two = 4 * tiles >= 3 * cus || (!p.offsets && p.rows > 128 && 2 * tiles > cus);
  if (epi == MP_EPI_SWIGLU)
    return two ? i8w_launch<MP_EPI_SWIGLU, 2, false>(p, 1, stream) : i8w_launch<MP_EPI_SWIGLU, 1, false>(p, 1, stream);
  if (epi == MP_EPI_F32) return two ? i8w_launch<MP_EPI_F32, 2, false>(p, 1, stream) : i8w_launch<MP_EPI_F32, 1, false>(p, 1, stream);
  return two ? i8w_launch<MP_EPI_DENSE, 2, false>(p, 1, stream) : i8w_launch<MP_EPI_DENSE, 1, false>(p, 1, stream);
}

int mp_i8_wide_splits(int64_t m, int64_t n, int64_t k) { return wide_splits(m, n, k); }

int mp_launch_i8_split(const mp_i8_args &p, int splits, int *partials, hipStream_t stream) {
  mp_i8_args d = p;
  d.y = partials;
  d.ldy = p.n;
  d.out_dtype = MP_F32;
  const int rc = i8w_launch<MP_EPI_DENSE, 1, true>(d, splits, stream);
  if (rc != MP_OK) return rc;
  const int64_t threads = p.rows * mp_cdiv(p.n, 4);
  hipLaunchKernelGGL(i8_reduce_kernel, dim3(static_cast<unsigned>(mp_cdiv(threads, 256))), dim3(256), 0, stream, partials,
                     splits, p);
  MP_CHECK_LAUNCH();
  return MP_OK;
}
