// W4A16 GEMM (group 128) for more rows than the streaming kernels take: activations and packed weights
// straight from memory into LDS, the weights dequantised in registers between the MFMAs.  The phases, the
// roles of the waves and the activation stages are dq_wide_kernel's (dqwide.hip).
//
// What bounds it: the fp16 / bf16 matrix cores at a few hundred rows, below that the weight stream and, per weight,
// about two VALU instructions.  Staging the dequantised tile through LDS instead (the prefill kernel) reads and
// writes four times the weight bytes there.
#include "w4_wide.h"
#include "wide_common.h"

#include <type_traits>

namespace {

// Eight nibbles of a packed word, column order, as r((u - z) s) in the dtype.  With h = 1024 + u (or 1024 + 16 u from
// the odd nibbles' place) in fp16, h s - (1024 + z) s (h s / 16 - (64 + z) s) in one fma is exact in fp32: both
// products have at most 22 significant bits (z an integer up to 15, an 11-bit s) and so has (u - z) s; one
// conversion rounds.
struct W4Scale {
  float s, s16, ne, no;  // s, s / 16, -(1024 + z) s, -(64 + z) s
};
template <int DT>
__device__ __forceinline__ uint4 w4w_dq8(uint32_t w, const W4Scale &c) {
  const uint32_t w8 = w >> 8;
  const whf2_t e0 = __builtin_bit_cast(whf2_t, (w & 0x000F000Fu) | 0x64006400u);
  const whf2_t o0 = __builtin_bit_cast(whf2_t, (w & 0x00F000F0u) | 0x64006400u);
  const whf2_t e1 = __builtin_bit_cast(whf2_t, (w8 & 0x000F000Fu) | 0x64006400u);
  const whf2_t o1 = __builtin_bit_cast(whf2_t, (w8 & 0x00F000F0u) | 0x64006400u);
  return make_uint4(
      wide_pack2<DT>(fmaf(static_cast<float>(e0[0]), c.s, c.ne), fmaf(static_cast<float>(o0[0]), c.s16, c.no)),
      wide_pack2<DT>(fmaf(static_cast<float>(e1[0]), c.s, c.ne), fmaf(static_cast<float>(o1[0]), c.s16, c.no)),
      wide_pack2<DT>(fmaf(static_cast<float>(e0[1]), c.s, c.ne), fmaf(static_cast<float>(o0[1]), c.s16, c.no)),
      wide_pack2<DT>(fmaf(static_cast<float>(e1[1]), c.s, c.ne), fmaf(static_cast<float>(o1[1]), c.s16, c.no)));
}

// Eight nibbles as u - z in fp16, column order; exact for a whole z up to 1024.
__device__ __forceinline__ uint4 w4w_sub8(uint32_t w, whf2_t z) {
  const uint32_t lo = w & 0xFFFFu, hi = w >> 16;
  const uint32_t a = (lo << 12) | lo, b = (hi << 12) | hi;  // nibbles 0 1 | 2 3 of each half at bits 0 and 16, 8 and 24 - 4
  const uint32_t p[4] = {a, a >> 8, b, b >> 8};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(whf2_t, (p[i] & 0x000F000Fu) | 0x64006400u) -
                                         whf2_t{1024, 1024}) - z);
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// The whole part of a zero point; the rest is exact in fp16.
__device__ __forceinline__ float w4w_whole(float z) { return fminf(fmaxf(rintf(z), -1024.f), 1024.f); }

template <int DT>
__device__ __forceinline__ float w4w_f32(uint32_t pair, int hi) {
  const uint16_t b = static_cast<uint16_t>(hi ? pair >> 16 : pair);
  return DT == MP_F16 ? mp_h2f(b) : mp_bf2f(b);
}

__device__ __forceinline__ void w4w_lds_load4(__amdgpu_buffer_rsrc_t r, int8_t *lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, reinterpret_cast<__attribute__((address_space(3))) void *>(reinterpret_cast<uintptr_t>(lds)), 4, voff,
      __builtin_amdgcn_readfirstlane(static_cast<int>(soff)), 0, 0);
}

// A workgroup of eight waves (two along M, four along N): up to 256 rows x BN = 128 TN weight rows (SwiGLU: BN / 2
// gate and the BN / 2 matching up rows).  LDS: three activation stages of K = 64 (128-byte rows, sized by the row
// tiles that are there), a ring of weight stages of K = 128 (64-byte rows, 16-byte chunk c of row r at slot
// c ^ ((r >> 2) & 3)) and two scale / zero stages of K = 256 (a lane's two groups in one 32-bit word).  A lane's
// 16-byte weight chunk is its K 32 h .. + 32 of a step (h = lane / 32): the four words are the operands of four MFMAs,
// whose activation chunks are 4 h + c.
//
// FACT (fp16): the operand is u - z and each group's sum is scaled in fp32, so no weight is rounded; the group's
// accumulators come on top of the totals, which leaves room for one column tile per wave.
//
// part (TN = 1): workgroup `sp` of `splits` takes that share of the 256-wide K stages and stores its fp32 sums to
// part[sp] for wide_reduce_kernel.
template <int DT, bool SWI, int TN, bool FACT>
__global__ __launch_bounds__(512, 2) void w4_wide_kernel(mp_w4_wide_args p, int n_slots, int splits, float *part) {
  constexpr int TM = 4, WN = 4, BN = 128 * TN;
  constexpr int QB = BN / 16 / 4;  // load instructions per weight stage of a loading wave
  constexpr int BST = BN * 64, SST = BN * 8;
  constexpr int CW = SWI ? 32 : 32 * TN;
  static_assert((!SWI || TN == 2) && (!FACT || (TN == 1 && !SWI && DT == MP_F16)), "forms");
  extern __shared__ __attribute__((aligned(16))) int8_t smem_w4[];
  const int bx = static_cast<int>(blockIdx.x);
  constexpr int CPT = SWI ? BN / 2 : BN;      // output columns of a tile
  const int64_t n_all = SWI ? p.n / 2 : p.n;  // output columns
  int col, slot, sp;
  const bool ok =
      wide_tile(bx, static_cast<int>((n_all + CPT - 1) / CPT), n_slots, TN == 1 ? splits : 1, false, col, slot, sp);
  const int64_t rb = static_cast<int64_t>(slot) * 256;
  if (!ok || rb >= p.m) return;  // a slot is below p.m / 256; without the test the compiler spills 35 registers of FACT
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, half = lane >> 5;
  const uint32_t k = static_cast<uint32_t>(p.k);
  const int rows = static_cast<int>(p.m - rb < 256 ? p.m - rb : 256);
  const int n_out = static_cast<int>(n_all), c0 = col * CPT;
  const int nt = (rows + 31) / 32;
  const int nv = nt > wm ? (nt - wm + 1) / 2 : 0;
  const int ast = nt * 32 * 128, s0 = 3 * ast, b0 = s0 + 2 * SST;
  const int nbs = min(6, (kWLds - (nt & 1) * 1024 - b0) / BST);

  const auto arsrc = mp_rsrc(p.x + rb * p.k, static_cast<uint32_t>(rows) * k * 2);
  const auto brsrc = mp_rsrc(p.w, static_cast<uint32_t>(p.n) * (k / 2));
  const uint32_t ng = k / 128;
  const auto srsrc = mp_rsrc(p.scales, static_cast<uint32_t>(p.n) * ng * 2);
  const auto zrsrc = mp_rsrc(p.zeros ? p.zeros : p.scales, static_cast<uint32_t>(p.n) * ng * 2);
  // activation loads (wave row 1): rows (4 q + wn) 8 .. + 8, lane l row l / 8, slot l % 8; weight loads (wave row 0): rows
  // (4 q + wn) 16 .. + 16, lane l row l / 4, slot l % 4
  uint32_t voff[8], szoff;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    if (wm == 1) {
      const int r = (q * 4 + wn) * 8 + lane / 8;
      voff[q] = r < rows ? static_cast<uint32_t>(r) * k * 2 + 16 * ((lane & 7) ^ ((r >> 1) & 7)) : kWOob;
    } else {
      const int r = (q * 4 + wn) * 16 + lane / 4;
      const int c = c0 + (SWI ? r % (BN / 2) : r);
      const uint32_t row = static_cast<uint32_t>(c + (SWI && r >= BN / 2 ? n_out : 0));
      voff[q] = c < n_out && r < BN ? row * (k / 2) + 16 * ((lane & 3) ^ ((r >> 2) & 3)) : kWOob;
    }
  }
  // scale / zero loads of wave row 0: 64 weight rows per wave (TN = 1: waves 2 and 3 repeat 0 and 1)
  {
    const int r = (TN == 2 ? wn : wn & 1) * 64 + lane;
    const int c = c0 + (SWI ? r % (BN / 2) : r);
    const uint32_t row = static_cast<uint32_t>(c + (SWI && r >= BN / 2 ? n_out : 0));
    szoff = c < n_out ? row * ng * 2 : kWOob;
  }
  int colj[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) colj[j] = c0 + (SWI ? wn * 32 : (wn * TN + j) * 32) + (lane & 31);

  // scale stages [first, first + nks), and their weight stages and K steps
  const int all = static_cast<int>(k / 256), first = TN == 1 ? all * sp / splits : 0;
  const int nks = TN == 1 ? all * (sp + 1) / splits - first : all, nkb = 2 * nks, nkt = 4 * nks;
  // XCDs start at different places of K (in units of a scale stage) and wrap around, see dq_wide_kernel
  const int rot = (bx & 7) * nks / 8;
  auto wrap = [](int t, int n) { return min(t < n ? t : t - n, n - 1); };
  auto load_a = [&](int kt, int slot, int q) {
    const int g = q * 4 + wn;
    wide_lds_load16(arsrc, smem_w4 + (g < nt * 4 ? slot * ast + g * 1024 : kWLds - 1024), voff[q],
                    (4 * first + wrap(kt + 4 * rot, nkt)) * (kWBK * 2));
  };
  auto load_b = [&](int kb, int slot, int q) {
    wide_lds_load16(brsrc, smem_w4 + b0 + slot * BST + (q * 4 + wn) * 1024, voff[q],
                    (2 * first + wrap(kb + 2 * rot, nkb)) * 64);
  };
  auto load_sz = [&](int ks) {  // two instructions
    int8_t *st = smem_w4 + s0 + (ks & 1) * SST + (TN == 2 ? wn : wn & 1) * 256;
    const uint32_t at = (first + wrap(ks + rot, nks)) * 4;
    w4w_lds_load4(srsrc, st, szoff, at);
    w4w_lds_load4(zrsrc, st + BN * 4, szoff, at);
  };
  auto wait_b = [&](int n, bool sz) {  // at most n weight stages (and the scale loads before the last) in flight
    if (n <= 0) wide_wait_vm<0>();
    else if (n == 1) { if (sz) wide_wait_vm<QB + 2>(); else wide_wait_vm<QB>(); }
    else if (n == 2) { if (sz) wide_wait_vm<2 * QB + 2>(); else wide_wait_vm<2 * QB>(); }
    else if (n == 3) { if (sz) wide_wait_vm<3 * QB + 2>(); else wide_wait_vm<3 * QB>(); }
    else { if (sz) wide_wait_vm<4 * QB + 2>(); else wide_wait_vm<4 * QB>(); }
  };

  f16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int aswz = (lane >> 1) & 7, bswz = (lane >> 2) & 3;
  const int abase = (wm * 32 + (lane & 31)) * 128;
  const int brow = (SWI ? wn * 32 : wn * TN * 32) + (lane & 31);  // the lane's weight row of column tile 0
  constexpr int BJ = SWI ? BN / 2 : 32;                           // rows to the next column tile's

  auto k_loop = [&](auto h_, auto nv_, auto wm_) {
    constexpr int H = decltype(h_)::value, NV = decltype(nv_)::value, WMC = decltype(wm_)::value;
    constexpr int KPH = H * TN > 6 ? 1 : 2;  // K = 32 or 64 per phase
    constexpr int NC = 2 * KPH;              // MFMA operands (words) per phase
    constexpr int NM = KPH * NV * TN;        // MFMAs of half a phase
    constexpr int VP = KPH * TN * 20 / (NM > 0 ? NM : 1) + 1;
    if constexpr (WMC == 1) {
#pragma unroll
      for (int st = 0; st < 3; ++st)
#pragma unroll
        for (int q = 0; q < 2 * H; ++q) load_a(st, st, q);
      wide_wait_vm<4 * H>();
    } else {
      load_sz(0);
      for (int st = 0; st < nbs - 1; ++st)
#pragma unroll
        for (int q = 0; q < QB; ++q) load_b(st, st, q);
      wait_b(nbs - 2, false);
    }
    wide_phase();
    if constexpr (WMC == 1) wide_phase();
    __builtin_amdgcn_s_waitcnt(kWLgkm0);  // only LDS reads are counted inside the loop
    int sa = 0, sb = 0;
    i4_t braw[TN];
    W4Scale cs[TN];
    f16_t grp[FACT ? (NV > 0 ? NV : 1) : 1];
    uint64_t rests = 0;  // FACT: lanes whose column has a zero point that is not whole
    // one K step of 64, P = kt % 4 (two steps to a group and a weight stage, four to a scale stage)
    auto step = [&](auto p_, int kt) {
      constexpr int P = decltype(p_)::value;
      const int8_t *pa = smem_w4 + sa * ast, *pb = smem_w4 + b0 + sb * BST, *ps = smem_w4 + s0 + ((kt >> 2) & 1) * SST;
#pragma unroll
      for (int k0 = 0; k0 < 2; k0 += KPH) {
        i4_t af[NC][NV > 0 ? NV : 1];
        uint4 bf[NC][TN];
        auto dequant = [&](int c) {
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if constexpr (FACT) {
              const _Float16 z = static_cast<_Float16>(cs[j].no);
              bf[c][j] = w4w_sub8(static_cast<uint32_t>(braw[j][2 * k0 + c]), whf2_t{z, z});
            } else {
              bf[c][j] = w4w_dq8<DT>(static_cast<uint32_t>(braw[j][2 * k0 + c]), cs[j]);
            }
          }
        };
        if constexpr (NV > 0) {
          uint32_t sp[TN], zp[TN];
          if (k0 == 0) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              const int r = brow + j * BJ;
              braw[j] = *reinterpret_cast<const i4_t *>(pb + r * 64 + 16 * ((2 * (P & 1) + half) ^ bswz));
              if ((P & 1) == 0) {
                sp[j] = *reinterpret_cast<const uint32_t *>(ps + r * 4);
                zp[j] = *reinterpret_cast<const uint32_t *>(ps + BN * 4 + r * 4);
              }
            }
          }
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < NV; ++i)
              af[c][i] = *reinterpret_cast<const i4_t *>(pa + abase + i * 2 * 32 * 128 +
                                                         16 * ((4 * half + 2 * k0 + c) ^ aswz));
          __builtin_amdgcn_sched_barrier(0);  // every read goes out before the dequantisation
          if (k0 == 0 && (P & 1) == 0) {
            if constexpr (FACT) {
              if (kt > 0) {  // the last group's sums
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                  for (int r = 0; r < 16; ++r) acc[i][0][r] = fmaf(grp[i][r], cs[0].s, acc[i][0][r]);
              }
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              const float s = w4w_f32<DT>(sp[j], P >> 1), z = p.zeros ? w4w_f32<DT>(zp[j], P >> 1) : 8.0f;
              if constexpr (FACT) {
                cs[j] = W4Scale{s, 0.f, 0.f, w4w_whole(z)};
                rests |= __ballot(cs[j].no != z);
              } else cs[j] = W4Scale{s, s * 0.0625f, -(1024.f + z) * s, -(64.f + z) * s};
            }
          }
#pragma unroll
          for (int c = 0; c < KPH; ++c) dequant(c);
        }
        if (WMC == 1 && k0 + KPH == 2) wide_wait_vm<2 * H>();  // the next step's activations have landed
        __builtin_amdgcn_s_waitcnt(kWLgkm0);
        wide_phase();
        __builtin_amdgcn_s_setprio(1);
        auto mma = [&](int c, int i, int j) {
          if constexpr (FACT) {
            const f16_t zero = {};
            grp[i] = wide_mfma<DT>(af[c][i], bf[c][j], (P & 1) == 0 && k0 == 0 && c == 0 ? zero : grp[i]);
          } else {
            acc[i][j] = wide_mfma<DT>(af[c][i], bf[c][j], acc[i][j]);
          }
        };
        if constexpr (NV > 0) {
#pragma unroll
          for (int c = KPH; c < NC; ++c) dequant(c);
#pragma unroll
          for (int x = 0; x < NM; ++x) mma(x / (NV * TN), x / TN % NV, x % TN);
#pragma unroll
          for (int x = 0; x < NM; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VP, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // loads into stages that every wave has read: activations three steps on, and on even steps the scales of
        // the next scale stage (once in four steps), then the last weight stage
        const bool loads = WMC == 1 ? k0 + KPH == 2 : ((P & 1) == 0 && k0 == 0);
        constexpr int QL = WMC == 1 ? 2 * H : QB + (P == 0 ? 1 : 0);
        auto load = [&](int q) {
          if (WMC == 1) load_a(kt + 3, sa, q);
          else if (P == 0 && q == 0) load_sz(kt / 4 + 1);
          else load_b(kt / 2 + nbs - 1, sb == 0 ? nbs - 1 : sb - 1, P == 0 ? q - 1 : q);
        };
        if constexpr (NV > 0) {
#pragma unroll
          for (int x = 0; x < NM; ++x) {
            mma(KPH + x / (NV * TN), x / TN % NV, x % TN);
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
        // the next weights (and on the last of four steps the next scales) have landed
        if (WMC == 0 && (P & 1) == 1 && k0 + KPH == 2) wait_b(P == 1 ? nbs - 2 : min(nbs - 2, 2), P == 1);
        wide_phase();
      }
      sa = sa == 2 ? 0 : sa + 1;
      if (P & 1) sb = sb == nbs - 1 ? 0 : sb + 1;
    };
    for (int kt = 0; kt < nkt; kt += 4) {
      step(std::integral_constant<int, 0>{}, kt);
      step(std::integral_constant<int, 1>{}, kt + 1);
      step(std::integral_constant<int, 2>{}, kt + 2);
      step(std::integral_constant<int, 3>{}, kt + 3);
    }
    if constexpr (FACT && NV > 0) {
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][0][r] = fmaf(grp[i][r], cs[0].s, acc[i][0][r]);
    }
    if constexpr (FACT && NV > 0) {
      // The loop took off whole zero points; what is left of them, which fp16 holds, is an operand of its own against
      // the activations, read again from memory.  (As a branch in the phases it cost 7% where no zero point has a
      // rest, or the registers: 208 spilled.)
      if (rests) {
        const int64_t cz = static_cast<int64_t>(min(colj[0], n_out - 1)) * ng + 2 * first;
#pragma unroll 1
        for (int g = 0; g < 2 * nks; ++g) {
          const float z = mp_h2f(p.zeros[cz + g]), s = mp_h2f(p.scales[cz + g]);
          const _Float16 d = static_cast<_Float16>(w4w_whole(z) - z);
          if (!__any(d != static_cast<_Float16>(0))) continue;
          const uint32_t dd = __builtin_bit_cast(uint32_t, whf2_t{d, d}), at = static_cast<uint32_t>(2 * first + g) * 256;
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            const int r = (i * 2 + wm) * 32 + (lane & 31);
            const uint32_t vo = r < rows ? static_cast<uint32_t>(r) * k * 2 + 16 * half : kWOob;
            f16_t t = {};
#pragma unroll 1
            for (uint32_t c = 0; c < 256; c += 32)
              t = wide_mfma<DT>(__builtin_bit_cast(i4_t, mp_buf_load16(arsrc, vo, at + c)), make_uint4(dd, dd, dd, dd), t);
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][0][q] = fmaf(t[q], s, acc[i][0][q]);
          }
        }
      }
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

  if constexpr (TN == 1) {
    if (part) {
      const int cj = c0 + wn * 32;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i >= nv) continue;  // wave-uniform
        const int lr = (i * 2 + wm) * 32;
        wide_store_part(acc[i][0], smem_w4 + wave * (32 * 144), part + (sp * p.m + rb + lr) * n_all + cj, n_all, rows - lr,
                        n_out - cj, lane);
      }
      return;
    }
  }
  // ---- epilogue: accumulator r of tile (i, j) is row 8 (r >> 2) + 4 half + (r & 3), column lane % 32
  float bv[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int c = (colj[j] < n_out ? colj[j] : n_out - 1) + (SWI && j ? n_out : 0);
    bv[j] = p.bias ? mp_load_as_f32(p.bias, c, DT) : 0.f;
  }
  const bool vec = n_out % 8 == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0;
  constexpr int LDR = CW * 2 + 16;
  int8_t *stage = smem_w4 + wave * (32 * LDR);
  const int cbase = c0 + (SWI ? wn * 32 : wn * TN * 32);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (i >= nv) continue;  // wave-uniform
    const int64_t m0 = rb + (i * 2 + wm) * 32;
#pragma unroll
    for (int j = 0; j < (SWI ? 1 : TN); ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        float v = mp_add(acc[i][j][r], bv[j]);
        if constexpr (SWI)
          v = mp_swiglu_epi(v, mp_add(acc[i][TN - 1][r], bv[TN - 1]), DT == MP_F16 ? kRoundF16 : kRoundBF16);
        const uint16_t o = DT == MP_F16 ? mp_f2h(v) : mp_f2bf(v);
        if (vec) *reinterpret_cast<uint16_t *>(stage + row * LDR + (j * 32 + (lane & 31)) * 2) = o;
        else if (m0 + row < p.m && colj[j] < n_out) p.y[(m0 + row) * n_all + colj[j]] = o;
      }
    if (!vec) continue;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int q = 0; q < CW / 16; ++q) {
      const int c = q * 64 + lane, row = c / (CW / 8), cc = (c % (CW / 8)) * 8;
      const uint4 v = *reinterpret_cast<const uint4 *>(stage + row * LDR + cc * 2);
      if (m0 + row < p.m && cbase + cc < n_out)
        *reinterpret_cast<uint4 *>(p.y + (m0 + row) * n_all + cbase + cc) = v;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the next tile overwrites the region
  }
}

template <int DT, bool SWI, int TN, bool FACT>
int w4w_launch(const mp_w4_wide_args &a, int splits, float *part, hipStream_t stream) {
  const int64_t slots = mp_cdiv(a.m, 256);
  const int64_t wgs = wide_grid(mp_cdiv(SWI ? a.n / 2 : a.n, SWI ? 64 * TN : 128 * TN), slots, splits, false);
  if (wgs > INT32_MAX) return MP_ERR_SHAPE;
  const void *fn = reinterpret_cast<const void *>(w4_wide_kernel<DT, SWI, TN, FACT>);
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kWLds) != hipSuccess) return MP_ERR_HIP;
  hipLaunchKernelGGL((w4_wide_kernel<DT, SWI, TN, FACT>), dim3(static_cast<unsigned>(wgs)), dim3(512),
                     kWLds, stream, a, static_cast<int>(slots), splits, part);
  MP_CHECK_LAUNCH();
  return part ? wide_reduce<DT>(part, splits, a.m, a.n, a.bias, a.y, stream) : MP_OK;
}

template <int DT>
int w4w_pick(const mp_w4_wide_args &a, bool swiglu, int splits, float *part, hipStream_t stream) {
  if (swiglu) return w4w_launch<DT, true, 2, false>(a, 1, nullptr, stream);
  const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256;
  const int64_t tiles = mp_cdiv(a.n, 256) * mp_cdiv(a.m, 256);
  if (!part && 4 * tiles >= 3 * cus) return w4w_launch<DT, false, 2, false>(a, 1, nullptr, stream);
  return w4w_launch<DT, false, 1, false>(a, splits, part, stream);
}

}  // namespace

bool mp_w4_wide_takes(const mp_w4_wide_args &a, bool swiglu) {
  // MP_W4_WIDE=0: the kernels before this one, for measurements
  static const bool on = !(mp_knob("MP_W4_WIDE") && atoi(mp_knob("MP_W4_WIDE")) == 0);
  return on && a.k % 256 == 0 && a.k <= (1 << 20) && a.n * (a.k / 2) < (int64_t(1) << 31) && mp_aligned(a.x, 16) &&
         mp_aligned(a.w, 16) && mp_aligned(a.scales, 4) && (!a.zeros || mp_aligned(a.zeros, 4)) && a.m > 0 &&
         a.m <= INT32_MAX && a.n <= INT32_MAX && (!swiglu || a.n % 2 == 0);
}

int mp_launch_w4_wide(const mp_w4_wide_args &a, bool swiglu, bool rounded, int splits, float *partials, hipStream_t stream) {
  if (!partials) splits = 1;
  if (a.dt == MP_BF16) return w4w_pick<MP_BF16>(a, swiglu, splits, partials, stream);
  if (rounded || swiglu) return w4w_pick<MP_F16>(a, swiglu, splits, partials, stream);
  return w4w_launch<MP_F16, false, 1, true>(a, splits, partials, stream);
}

// SwiGLU (a workgroup makes 128 output columns of up to 256 rows): from more than half of the CUs, where the prefill
// kernel's workgroups of half the size come to more than one round (M = 768, 2 I = 11264, K = 2048 (132 workgroups) 61
// against 88 us, M = 300, 2 I = 22016, K = 4096 93 against 144 us, M = 2048 354 against 475 us); below that the kernels
// before it are faster (M = 65, 2 I = 12288, K = 4096 in bf16 62 against 35 us, M = 256, 2 I = 22016 93 against 78 us,
// M = 512, 2 I = 16384 94 against 85 us), as at K = 1024 with a second round of up to half the CUs (M = 1536, 2 I =
// 14336 88 against 82 us).
//
// Linears from 96 tiles of 256 rows x 128 columns.  Against the prefill kernel (M = 2048, N = 12288 230 against 265 us,
// M = 512, N = 22016 126 against 152 us, M = 600, 8192 x 8192 112 against 153 us, M = 128, N = 28672, K = 8192 93
// against 133 us; with 32 tiles 56 against 33 us) from K = 1024: below it a tile's start and end count for more (M =
// 1024, N = 20480, K = 256 43 against 32 us, K = 512 53 against 44 us), at 1024 not in a second round of up to half the
// CUs (M = 768, N = 24576 74 against 69 us), nor up to 128 rows from three quarters of the CUs' 256-column tiles (M =
// 128, N = 65536 32.4 against 29.7 us), nor, below 4096, up to 128 rows with a second round of 128-column tiles on less
// than half of the CUs (M = 128, N = 40960, K = 2048 51 against 45 us).  Against the batched kernel's row parts only in
// fp16, in one row slot and from K = 2048 (M = 128, N = 12288, K = 2048 in fp16 / bf16 19.0 / 22.9 against 20.0 / 20.6
// us, K = 1024 15.0 against 12.2 us, M = 128, N = 16384, K = 2048 24 against 20 us, M = 300, N = 6144, K = 2048 31.8
// against 21.7 us), and below K = 1024, where those are slow (M = 128, N = 16384, K = 256 8.6 against 11.9 us), but for
// a second slot of a few rows.
bool mp_w4_wide_rule(const mp_w4_wide_args &a, bool swiglu) {
  if (a.m <= 64) return false;
  const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256, slots = mp_cdiv(a.m, 256);
  const int64_t tiles = mp_cdiv(a.n, 128) * slots, wide = mp_cdiv(a.n, 256) * slots;
  const bool short_tail = a.k < 2048 && wide > cus && 2 * wide <= 3 * cus;
  if (swiglu) return 2 * wide > cus && a.k >= 1024 && !short_tail;
  if (tiles < 96) return false;
  if (mp_w4_batch_numerics(a.m, a.n)) {
    if (a.k < 1024) return a.m <= 256 || tiles >= 128 || (a.m - 1) % 256 >= 127;
    return a.dt == MP_F16 && a.k >= 2048 && a.m <= 256 && (a.m < 128 || tiles < 128);
  }
  if (a.m <= 128 && a.k < 4096 && tiles > cus && 2 * tiles < 3 * cus) return false;
  return a.k >= 1024 && !short_tail && (a.k >= 2048 || a.m > 128 || 4 * wide < 3 * cus);
}

// K split from 2^32 multiply-adds, up to 256 rows below K = 4096 above them (less is what the second launch costs):
// measured against the batched kernel M = 77, N = 13824, K = 5120 36 against 55 us, M = 256, N = 4096, K = 11008 / 4096
// 41 / 29 against 85 / 33 us, M = 64, N = 8192, K = 28672 76 against 85 us; M = 65, 4096 x 4096 24 against 18 us, M =
// 256, N = 8192, K = 2048 28 against 23 us.
extern "C" size_t mp_w4a16_gemm_workspace_bytes(int64_t m, int64_t n, int64_t k, int group_size) {
  if (m <= 32 || m >= 1024 || n <= 0 || k <= 0 || group_size != 128 || k % 256 != 0) return 0;
  if (k > (1 << 20) || n > INT32_MAX || m * n < (int64_t(1) << 32) / k + (m <= 256 && k < 4096)) return 0;
  const int s = wide_splits(m, n, k);
  return s < 2 ? 0 : static_cast<size_t>(s) * static_cast<size_t>(m) * static_cast<size_t>(n) * sizeof(float);
}

extern "C" int mp_w4a16_gemm_ws(const void *x, int64_t m, int64_t k, const int32_t *w_packed, int64_t n,
                                const void *scales, const void *zeros, int group_size, const void *bias, void *y,
                                int x_dtype, void *workspace, size_t workspace_bytes, mp_stream_t stream) {
  const size_t need = mp_w4a16_gemm_workspace_bytes(m, n, k, group_size);
  const mp_w4_wide_args a{static_cast<const uint16_t *>(x), reinterpret_cast<const uint32_t *>(w_packed),
                          static_cast<const uint16_t *>(scales), static_cast<const uint16_t *>(zeros),
                          static_cast<const uint16_t *>(bias), static_cast<uint16_t *>(y), x_dtype, m, n, k};
  // fp16, two ways, up to 48 rows on less than three quarters of the CUs or up to 64 at K <= 4096: the batched kernel
  // (M = 40, N = 11008, K = 11008 52.5 against 47.1 us, K = 28672 level, in bf16 the split, 47 against 50 us; M = 64, N
  // = 16384, K = 4096 27 against 23.5 us, in bf16 the split, 25.6 against 32 us)
  const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256;
  const bool few = x_dtype == MP_F16 && need > 0 && wide_splits(m, n, k) == 2 &&
                   ((m <= 48 && 8 * mp_cdiv(n, 128) < 3 * cus) || (m <= 64 && k <= 4096));
  if (need == 0 || few || !workspace || workspace_bytes < need || !mp_aligned(workspace, 16) || !x || !w_packed || !scales ||
      !y || (x_dtype != MP_F16 && x_dtype != MP_BF16) || !mp_w4_wide_takes(a, false))
    return mp_w4a16_gemm(x, m, k, w_packed, n, scales, zeros, group_size, bias, y, x_dtype, stream);
  return mp_launch_w4_wide(a, false, !mp_w4_batch_numerics(m, n), wide_splits(m, n, k), static_cast<float *>(workspace),
                           reinterpret_cast<hipStream_t>(stream));
}
