// The dequantising GEMM for plain 16-bit activations and int8 weight rows: Y = A . r(q * s)^T, dense or
// grouped by expert, with the activations (and the fake-quant values among them) already rounded to the
// dtype.  The element rounding and the products are those of dq_gemm_kernel (dqgemm.hip).
//
// What bounds it: at a few hundred rows per weight the fp16 / bf16 matrix cores, below that the weight
// stream.  Both operands go straight from memory into LDS (`buffer_load ... lds`): no staging registers,
// the next stages in flight while one is multiplied.  The weights stay int8 in LDS (half the bytes of the
// dequantised tile) and a wave dequantises its own columns after reading them, 2.5 VALU instructions per
// weight, while the other wave of its SIMD feeds the matrix cores.
//
// Measured against dq_gemm_kernel with the codes as activations (module calls with the fake quant, random data):
// M = 1000, N = 13824, K = 5120 in bf16 226 -> 149 us (at 1.0 PFLOP/s the card is at its power limit: the MFMAs
// alone, on registers, take 88 us, with operands from LDS 110, with the dequantisation 120); the Mixtral-shaped
// experts (8 x 4096 x 14336, 512 tokens, top-2) 880 -> 566 us; M = 8, N = 11008, K = 4096 64 -> 12.6 us.
#include "dq_wide.h"
#include "wide_common.h"

namespace {

// 8 int8 codes times the row scale, rounded to the dtype (q * s: one fp32 product, one conversion).
template <int DT>
__device__ __forceinline__ uint4 wide_dq8(uint32_t w0, uint32_t w1, float s) {
  const uint32_t w[2] = {w0, w1};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float f0 = static_cast<float>(static_cast<int8_t>(w[i] & 0xFFu)) * s;
    const float f1 = static_cast<float>(static_cast<int8_t>((w[i] >> 8) & 0xFFu)) * s;
    const float f2 = static_cast<float>(static_cast<int8_t>((w[i] >> 16) & 0xFFu)) * s;
    const float f3 = static_cast<float>(static_cast<int8_t>(w[i] >> 24)) * s;
    o[2 * i] = wide_pack2<DT>(f0, f1);
    o[2 * i + 1] = wide_pack2<DT>(f2, f3);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// A workgroup of eight waves (two along M, four along N) makes a tile of up to 256 rows x BN = 128 TN weight rows
// (SwiGLU: BN / 2 gate rows and the BN / 2 up rows of the same output columns), a wave up to 4 x TN MFMA
// 32x32x16 tiles: row tiles 2 i + wm, interleaved so that a partly filled tile (the last rows of an expert)
// splits evenly over the two waves of a SIMD; H = ceil(row tiles / 2) of wave row 0's tiles and NV of this wave's
// hold rows, the others are neither loaded nor multiplied.
//
// LDS: three activation stages of K = 64, sized by the row tiles that are there, and as many weight stages of
// K = 128 as the rest holds (2 at 192 rows and more with TN = 2, 3 up to 160 rows, 4 up to 64), both of
// 128-byte rows (a load instruction then reads 8 rows x 128 bytes; 16 rows x 64 bytes cost the CU half as
// much again), 16-byte chunk c of row r at slot c ^ ((r >> 1) & 7): the 16 rows of a ds_read_b128 quarter hit
// 16 distinct 16-byte bank groups.  A lane's 16-byte weight chunk holds K 32 kp + 16 h .. + 16 (h = lane / 32) of
// the step, the operand of two MFMAs; the activation chunks 4 kp + 2 h + m match that order of K.
//
// The K loop runs in phases that end at a barrier.  Waves 0..3 and 4..7, one of each on every SIMD, are one
// phase apart: while one reads its operands from LDS and dequantises half of its weights, the other
// multiplies, with the other half's dequantisation and the loads of later stages between its MFMAs (issued in
// the reading phase, those loads held it up: 100 -> 85 us for 16 tiles of 256 x 256 x 4096).  Waves 0..3
// load the weights and waves 4..7 the activations: loads complete in order, so a wave that waits for
// activations from L2 would wait for the weights it asked HBM for before them.  A phase is K = 64 where the
// registers hold its operands, else K = 32.
template <int DT, int EPI, int TN>
__global__ __launch_bounds__(512, 2) void dq_wide_kernel(mp_dq_args p, int n_slots, int splits, float *part) {
  constexpr bool SWI = EPI == MP_EPI_SWIGLU;
  constexpr int TM = 4, WM = 2, WN = 4, BN = 128 * TN;
  constexpr int QB = BN / 8 / 4;  // load instructions per weight stage of a loading wave
  constexpr int BST = BN * 128;
  constexpr int CW = SWI ? 32 : 32 * TN;  // output columns of a wave
  static_assert(!SWI || TN == 2, "gate and up tiles meet in one wave");
  extern __shared__ __attribute__((aligned(16))) int8_t smem_wide[];
  const int bx = static_cast<int>(blockIdx.x);
  constexpr int CPT = SWI ? BN / 2 : BN;  // output columns of a tile
  int col, slot, sp;
  if (!wide_tile(bx, static_cast<int>((p.n + CPT - 1) / CPT), n_slots, TN == 1 ? splits : 1,
                 wide_by_slot(p.offsets, p.n_experts, n_slots), col, slot, sp))
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
  const int nt = (rows + 31) / 32;               // row tiles that hold rows
  const int nv = nt > wm ? (nt - wm + 1) / 2 : 0;  // this wave's
  const int ast = nt * 32 * 128, b0 = 3 * ast;
  // weight stages; with an odd nt the last kilobyte takes the loads of the row groups that pad it to an even one
  const int nbs = min(TN == 2 ? 4 : 6, (kWLds - (nt & 1) * 1024 - b0) / BST);

  const auto arsrc = mp_rsrc(static_cast<const uint16_t *>(p.a) + rb * p.k, static_cast<uint32_t>(rows) * k * 2);
  const auto brsrc = mp_rsrc(static_cast<const int8_t *>(p.b) + expert * nb_rows * p.k,
                             static_cast<uint32_t>(nb_rows) * k);
  // load instruction q of the wave: rows (4 q + wn) 8 .. + 8 of the stage, lane l row l / 8, slot l % 8
  uint32_t voff[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = (q * 4 + wn) * 8 + lane / 8;
    const uint32_t ch = 16 * ((lane & 7) ^ ((r >> 1) & 7));
    if (wm == 1) {
      voff[q] = r < rows ? static_cast<uint32_t>(r) * k * 2 + ch : kWOob;
    } else {
      const int c = c0 + (SWI ? r % (BN / 2) : r);
      const uint32_t row = static_cast<uint32_t>(c + (SWI && r >= BN / 2 ? n_out : 0));
      voff[q] = c < n_out && r < BN ? row * k + ch : kWOob;
    }
  }
  float bs[TN];
  int colj[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    colj[j] = c0 + (SWI ? wn * 32 : (wn * TN + j) * 32) + (lane & 31);
    const int c = colj[j] < n_out ? colj[j] : n_out - 1;
    bs[j] = p.b_scale[expert * nb_rows + c + (SWI ? j * p.n : 0)];
  }
  // K steps [first, first + nkt) and their weight stages (a split starts and ends at a weight stage)
  const int all = static_cast<int>(k / kWBK), first = TN == 1 ? all / 2 * sp / splits * 2 : 0;
  const int nkt = (TN == 1 && sp + 1 < splits ? all / 2 * (sp + 1) / splits * 2 : all) - first, nkb = (nkt + 1) / 2;
  // XCDs and experts start at different places of K and wrap around: in step, every workgroup would ask for the same
  // 128 bytes of rows that lie K bytes apart, which at K = 4096 is a few of the memory channels at a time (32 rows,
  // 65536 x 4096, a start of its own for each column tile: 74 -> 59 us).  The workgroups of an XCD that share
  // activation rows stay in step: the experts' rows together exceed its L2.  An odd number of steps starts at 0: its
  // last weight stage's second half is the next row's bytes (or, past the buffer, zeros) and never read.  Stages past
  // the end are loaded and never read.
  const int rot = nkt & 1 ? 0 : ((bx & 7) * nkb / 8 + expert * 5) % nkb;
  auto wrap = [](int t, int n) { return min(t < n ? t : t - n, n - 1); };
  auto load_a = [&](int kt, int slot, int q) {
    const int g = q * 4 + wn;  // 8-row group
    wide_lds_load16(arsrc, smem_wide + (g < nt * 4 ? slot * ast + g * 1024 : kWLds - 1024), voff[q],
                    (first + wrap(kt + 2 * rot, nkt)) * (kWBK * 2));
  };
  auto load_b = [&](int kb, int slot, int q) {
    wide_lds_load16(brsrc, smem_wide + b0 + slot * BST + (q * 4 + wn) * 1024, voff[q],
                    (first + 2 * wrap(kb + rot, nkb)) * kWBK);
  };
  // at most n weight stages still in flight
  auto wait_b = [&](int n) {
    if (n <= 0) wide_wait_vm<0>();
    else if (n == 1) wide_wait_vm<QB>();
    else if (n == 2) wide_wait_vm<2 * QB>();
    else if (n == 3) wide_wait_vm<3 * QB>();
    else wide_wait_vm<4 * QB>();
  };

  f16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int swz = (lane >> 1) & 7;
  const int abase = (wm * 32 + (lane & 31)) * 128;
  const int bbase = b0 + ((SWI ? wn * 32 : wn * TN * 32) + (lane & 31)) * 128;

  auto k_loop = [&](auto h_, auto nv_, auto wm_) {
    constexpr int H = decltype(h_)::value, NV = decltype(nv_)::value, WMC = decltype(wm_)::value;
    constexpr int KPH = H * TN > 6 ? 1 : 2;         // K = 32 or 64 per phase
    constexpr int NM = KPH * NV * TN;               // MFMAs of half a phase
    constexpr int VP = KPH * TN * 20 / (NM > 0 ? NM : 1) + 1;  // VALU instructions per MFMA that dequantise half of the weights
    constexpr int QL = WMC == 1 ? 2 * H : QB;       // loads of a step
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
    int sa = 0, sb = 0;                   // activation stage of the step, weight stage of the step pair
    // one K step of 64: PAR = 0 the first, 1 the second half of a weight stage
    auto step = [&](auto par_, int kt) {
      constexpr int PAR = decltype(par_)::value;
      const int8_t *pa = smem_wide + sa * ast, *pb = smem_wide + sb * BST;
#pragma unroll
      for (int k0 = 0; k0 < 2; k0 += KPH) {
        i4_t braw[KPH][TN], af[2 * KPH][NV > 0 ? NV : 1];
        uint4 bf[2 * KPH][TN];
        auto dequant = [&](int c) {  // operand c of the phase (K = 16)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            bf[c][j] = wide_dq8<DT>(braw[c / 2][j][2 * (c % 2)], braw[c / 2][j][2 * (c % 2) + 1], bs[j]);
        };
        if constexpr (NV > 0) {
#pragma unroll
          for (int kp = 0; kp < KPH; ++kp)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              braw[kp][j] = *reinterpret_cast<const i4_t *>(pb + bbase + j * (SWI ? BN / 2 : 32) * 128 +
                                                            16 * ((4 * PAR + 2 * (k0 + kp) + half) ^ swz));
#pragma unroll
          for (int c = 0; c < 2 * KPH; ++c)
#pragma unroll
            for (int i = 0; i < NV; ++i)
              af[c][i] = *reinterpret_cast<const i4_t *>(pa + abase + i * 2 * 32 * 128 +
                                                         16 * ((4 * (k0 + c / 2) + 2 * half + c % 2) ^ swz));
          __builtin_amdgcn_sched_barrier(0);  // every read goes out before the dequantisation
#pragma unroll
          for (int c = 0; c < KPH; ++c) dequant(c);
        }
        // the next step's activations have landed (the barrier makes that every wave's)
        if (WMC == 1 && k0 + KPH == 2) wide_wait_vm<2 * H>();
        __builtin_amdgcn_s_waitcnt(kWLgkm0);
        wide_phase();
        __builtin_amdgcn_s_setprio(1);
        if constexpr (NV > 0) {
#pragma unroll
          for (int c = KPH; c < 2 * KPH; ++c) dequant(c);
#pragma unroll
          for (int x = 0; x < NM; ++x) {
            const int c = x / (NV * TN), i = x / TN % NV, j = x % TN;
            acc[i][j] = wide_mfma<DT>(af[c][i], bf[c][j], acc[i][j]);
          }
#pragma unroll
          for (int x = 0; x < NM; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VP, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // loads into stages that every wave has read: the activations three steps on, into the stage just
        // read (wave row 1 reads it last), and on even steps the last weight stage, read before this step
        const bool loads = WMC == 1 ? k0 + KPH == 2 : (PAR == 0 && k0 == 0);
        auto load = [&](int q) {
          if (WMC == 1) load_a(kt + 3, sa, q);
          else load_b(kt / 2 + nbs - 1, sb == 0 ? nbs - 1 : sb - 1, q);
        };
        if constexpr (NV > 0) {
#pragma unroll
          for (int x = 0; x < NM; ++x) {
            const int c = KPH + x / (NV * TN), i = x / TN % NV, j = x % TN;
            acc[i][j] = wide_mfma<DT>(af[c][i], bf[c][j], acc[i][j]);
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
        if (WMC == 0 && PAR == 1 && k0 + KPH == 2) wait_b(nbs - 2);  // the next pair's weights have landed
        wide_phase();
      }
      sa = sa == 2 ? 0 : sa + 1;
    };
    for (int kt = 0; kt < nkt; kt += 2) {
      step(std::integral_constant<int, 0>{}, kt);
      if (kt + 1 < nkt) step(std::integral_constant<int, 1>{}, kt + 1);
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

  if constexpr (TN == 1) {
    if (part) {
      const int cj = c0 + wn * 32;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if (i >= nv) continue;  // wave-uniform
        const int lr = (i * 2 + wm) * 32;
        wide_store_part(acc[i][0], smem_wide + wave * (32 * 144), part + (sp * p.rows + rb + lr) * p.n + cj, p.n, rows - lr,
                        n_out - cj, lane);
      }
      return;
    }
  }
  // ---- epilogue: accumulator r of tile (i, j) is row 8 (r >> 2) + 4 half + (r & 3), column lane % 32
  float bv[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    bv[j] = (!SWI && p.bias) ? mp_load_as_f32(p.bias, colj[j] < n_out ? colj[j] : n_out - 1, p.bias_dtype) : 0.f;
  const bool vec = p.out_dtype != MP_F32 && n_out % 8 == 0 && p.ldy % 8 == 0 &&
                   (reinterpret_cast<uintptr_t>(p.y) & 15) == 0;
  // 16-bit outputs through a wave-private LDS tile of 32 rows, then 16-byte stores
  constexpr int LDR = CW * 2 + 16;
  int8_t *stage = smem_wide + wave * (32 * LDR);
  const int cbase = c0 + (SWI ? wn * 32 : wn * TN * 32);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (i >= nv) continue;  // wave-uniform
    const int64_t m0 = rb + (i * WM + wm) * 32;
#pragma unroll
    for (int j = 0; j < (SWI ? 1 : TN); ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        const float v = SWI ? mp_swiglu_epi(acc[i][0][r], acc[i][TN - 1][r], DT == MP_F16 ? kRoundF16 : kRoundBF16)
                            : mp_add(acc[i][j][r], bv[j]);
        if (vec) {
          *reinterpret_cast<uint16_t *>(stage + row * LDR + (j * 32 + (lane & 31)) * 2) =
              p.out_dtype == MP_F16 ? mp_f2h(v) : mp_f2bf(v);
        } else if (m0 + row < re && colj[j] < n_out) {
          mp_store_from_f32(p.y, (m0 + row) * p.ldy + colj[j], p.out_dtype, v);
        }
      }
    if (!vec) continue;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int q = 0; q < CW / 16; ++q) {
      const int c = q * 64 + lane, row = c / (CW / 8), cc = (c % (CW / 8)) * 8;
      const uint4 v = *reinterpret_cast<const uint4 *>(stage + row * LDR + cc * 2);
      if (m0 + row < re && cbase + cc < n_out)
        *reinterpret_cast<uint4 *>(static_cast<uint16_t *>(p.y) + (m0 + row) * p.ldy + cbase + cc) = v;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the next tile overwrites the region
  }
}

template <int DT, int EPI, int TN>
int wide_launch(const mp_dq_args &p, int splits, float *part, hipStream_t stream) {
  const int64_t slots = wide_row_slots(p.rows, p.offsets ? p.n_experts : 1);
  const int64_t wgs = wide_grid(mp_cdiv(p.n, EPI == MP_EPI_SWIGLU ? 64 * TN : 128 * TN), slots, splits,
                                wide_by_slot(p.offsets, p.n_experts, slots));
  if (wgs > INT32_MAX) return MP_ERR_SHAPE;
  const void *fn = reinterpret_cast<const void *>(dq_wide_kernel<DT, EPI, TN>);
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kWLds) != hipSuccess) return MP_ERR_HIP;
  hipLaunchKernelGGL((dq_wide_kernel<DT, EPI, TN>), dim3(static_cast<unsigned>(wgs)), dim3(512), kWLds,
                     stream, p, static_cast<int>(slots), splits, part);
  MP_CHECK_LAUNCH();
  return part ? wide_reduce<DT>(part, splits, p.rows, p.n, p.bias, p.y, stream) : MP_OK;
}

// 256 weight rows per workgroup where that makes a tile for three quarters of the CUs (half the activation reads
// of 128 rows), else 128: M = 1000, N = 13824, K = 5120 (216 tiles) 134 against 159 us; M = 160, N = 32768,
// K = 14336 (128 tiles) 217 against 190 us; M = 256, 4096 x 4096 (16 tiles) 92 against 55 us.  Grouped: counted
// as if the rows were spread over all experts.
template <int DT, int EPI>
int wide_pick(const mp_dq_args &p, hipStream_t stream) {
  if constexpr (EPI == MP_EPI_SWIGLU) {
    return wide_launch<DT, EPI, 2>(p, 1, nullptr, stream);
  } else {
    const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256;
    const int64_t groups = p.offsets ? (p.rows < p.n_experts ? p.rows : p.n_experts) : 1;
    const int64_t tiles = mp_cdiv(p.n, 256) * groups * mp_cdiv(mp_cdiv(p.rows, groups), 256);
    if (4 * tiles >= 3 * cus) return wide_launch<DT, EPI, 2>(p, 1, nullptr, stream);
    return wide_launch<DT, EPI, 1>(p, 1, nullptr, stream);
  }
}

// ------------------------------------------------------------------ a few rows (M <= 32)
// What bounds it: the weight stream.  A workgroup of four waves per 16 NCT weight rows, each wave a contiguous quarter
// of K in steps of 128, streaming its activation rows (16 MT, 256 bytes a step) and the workgroup's weight
// rows into a ring of S LDS stages of its own by `buffer_load ... lds`, S - 1 steps ahead: no barrier in the K
// loop, and the activations are read once per workgroup.  MFMA 16x16x32; a lane's 16-byte weight chunk
// (K 64 ks + 16 q .. + 16, q = lane / 16) is dequantised in registers into the operands of two, whose
// activation chunks are 8 ks + 2 q + m.  16-byte chunk c of activation row r sits at slot c ^ (r & 15), of a weight
// row at c ^ ((r >> 1) & 7): conflict-free reads.  Rows past M and N lie past their descriptors (zeros, no
// memory access).  Column tiles start at different steps of each wave's range and wrap around (see
// dq_wide_kernel).  The four waves' fp32 sums meet in LDS and are added in wave order.
template <int MT, int NCT>
struct SkinnyShape {
  static constexpr int QA = 4 * MT, QB = 2 * NCT, STAGE = MT * 4096 + NCT * 2048;
  static constexpr int S = STAGE * 12 <= kWLds ? 3 : 2;
  static constexpr int SMEM = STAGE * S * 4 > MT * NCT * 4096 ? STAGE * S * 4 : MT * NCT * 4096;
  static_assert(SMEM <= kWLds, "stages");
};

template <int DT>
__device__ __forceinline__ f4_t wide_mfma16(i4_t a, uint4 b, f4_t c) {
  if constexpr (DT == MP_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a), __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wbf8_t, a), __builtin_bit_cast(wbf8_t, b), c, 0, 0,
                                                   0);
}

template <int DT, int MT, int NCT>
__global__ __launch_bounds__(256) void dq_skinny_kernel(mp_dq_args p) {
  using Sh = SkinnyShape<MT, NCT>;
  constexpr int S = Sh::S, QA = Sh::QA, QB = Sh::QB, QW = QA + QB;
  extern __shared__ __attribute__((aligned(16))) int8_t smem_skinny[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int8_t *ring = smem_skinny + wave * S * Sh::STAGE;
  const uint32_t k = static_cast<uint32_t>(p.k);
  const int rows = static_cast<int>(p.rows), n_out = static_cast<int>(p.n), c0 = static_cast<int>(blockIdx.x) * 16 * NCT;
  const auto arsrc = mp_rsrc(p.a, static_cast<uint32_t>(rows) * k * 2);
  const auto brsrc = mp_rsrc(static_cast<const int8_t *>(p.b) + static_cast<int64_t>(c0) * p.k,
                             static_cast<uint32_t>(min(n_out - c0, 16 * NCT)) * k);
  const int nst = static_cast<int>(k / 128);
  const int s0 = nst * wave / 4, len = nst * (wave + 1) / 4 - s0;  // this wave's steps: at least one (K >= 512)
  const int rot = static_cast<int>(blockIdx.x * 5u % static_cast<uint32_t>(len));
  uint32_t voff[QW];
#pragma unroll
  for (int q = 0; q < QA; ++q) {
    const int r = 4 * q + lane / 16;
    voff[q] = r < rows ? static_cast<uint32_t>(r) * k * 2 + 16 * ((lane & 15) ^ (r & 15)) : kWOob;
  }
#pragma unroll
  for (int q = 0; q < QB; ++q) {
    const int r = 8 * q + lane / 8;
    voff[QA + q] = c0 + r < n_out ? static_cast<uint32_t>(r) * k + 16 * ((lane & 7) ^ ((r >> 1) & 7)) : kWOob;
  }
  float bs[NCT];
#pragma unroll
  for (int j = 0; j < NCT; ++j) {
    const int c = c0 + 16 * j + (lane & 15);
    bs[j] = p.b_scale[c < n_out ? c : n_out - 1];
  }
  auto issue = [&](int t, int slot) {  // step t of the wave's range; past its end a step again, never read
    t = (t < len ? t : len - 1) + rot;
    const uint32_t at = static_cast<uint32_t>(s0 + (t < len ? t : t - len));
    int8_t *st = ring + slot * Sh::STAGE;
#pragma unroll
    for (int q = 0; q < QA; ++q) wide_lds_load16(arsrc, st + q * 1024, voff[q], at * 256);
#pragma unroll
    for (int q = 0; q < QB; ++q) wide_lds_load16(brsrc, st + MT * 4096 + q * 1024, voff[QA + q], at * 128);
  };
  f4_t acc[NCT][MT];
#pragma unroll
  for (int j = 0; j < NCT; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[j][t] = f4_t{0.f, 0.f, 0.f, 0.f};
  const int row = lane & 15, kq = lane >> 4, bswz = (lane >> 1) & 7;
#pragma unroll
  for (int s = 0; s < S - 1; ++s) issue(s, s);
  int slot = 0;
  for (int t = 0; t < len; ++t) {
    // own loads of the step landed (later steps' may remain) and own reads of the slot refilled next are done
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * QW) : "memory");
    issue(t + S - 1, slot == 0 ? S - 1 : slot - 1);
    const int8_t *st = ring + slot * Sh::STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      i4_t braw[NCT], af[2][MT];
#pragma unroll
      for (int j = 0; j < NCT; ++j)
        braw[j] = *reinterpret_cast<const i4_t *>(st + MT * 4096 + (16 * j + row) * 128 + 16 * ((4 * ks + kq) ^ bswz));
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t2 = 0; t2 < MT; ++t2)
          af[m][t2] = *reinterpret_cast<const i4_t *>(st + (16 * t2 + row) * 256 + 16 * ((8 * ks + 2 * kq + m) ^ row));
#pragma unroll
      for (int j = 0; j < NCT; ++j)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const uint4 bf = wide_dq8<DT>(braw[j][2 * m], braw[j][2 * m + 1], bs[j]);
#pragma unroll
          for (int t2 = 0; t2 < MT; ++t2) acc[j][t2] = wide_mfma16<DT>(af[m][t2], bf, acc[j][t2]);
        }
    }
    slot = slot == S - 1 ? 0 : slot + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS load in flight past this point
  mp_lds_barrier();                                 // every ring is done: reuse LDS for the sums
  float *red = reinterpret_cast<float *>(smem_skinny);  // [4][NCT * MT][4][64]
#pragma unroll
  for (int j = 0; j < NCT; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((wave * NCT * MT + j * MT + t) * 4 + i) * 64 + lane] = acc[j][t][i];
  mp_lds_barrier();
  for (int o = tid; o < NCT * MT * 256; o += 256) {
    const int jt = o >> 8, l = o & 63, i = (o >> 6) & 3;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) v = mp_add(v, red[((w * NCT * MT + jt) * 4 + i) * 64 + l]);
    const int m = (jt % MT) * 16 + 4 * (l >> 4) + i, col = c0 + (jt / MT) * 16 + (l & 15);
    if (m < rows && col < n_out) {
      if (p.bias) v = mp_add(v, mp_load_as_f32(p.bias, col, p.bias_dtype));
      mp_store_from_f32(p.y, m * p.ldy + col, p.out_dtype, v);
    }
  }
}

// Column tiles per workgroup: the fewest (1 to 4) that leave at most one workgroup per CU, so that each reads the
// activations once per CU; beyond that the most.
template <int DT, int MT>
int skinny_launch(const mp_dq_args &p, hipStream_t stream) {
  const int64_t cus = mp_cu_count() > 0 ? mp_cu_count() : 256;
  int nct = 1;
  while (nct < 4 && mp_cdiv(p.n, 16 * nct) > cus) ++nct;
#define MP_DQS(NCT_)                                                                                                  \
  do {                                                                                                                \
    constexpr int smem = SkinnyShape<MT, NCT_>::SMEM;                                                                 \
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(dq_skinny_kernel<DT, MT, NCT_>),                           \
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess)                          \
      return MP_ERR_HIP;                                                                                              \
    hipLaunchKernelGGL((dq_skinny_kernel<DT, MT, NCT_>), dim3(static_cast<unsigned>(mp_cdiv(p.n, 16 * NCT_))), dim3(256), \
                       smem, stream, p);                                                                              \
  } while (0)
  if (nct == 1) MP_DQS(1);
  else if (nct == 2) MP_DQS(2);
  else if (nct == 3) MP_DQS(3);
  else MP_DQS(4);
#undef MP_DQS
  MP_CHECK_LAUNCH();
  return MP_OK;
}

// The fake-quantized rows themselves, r(q * s) in the dtype, of the per-token 8-bit rule (mp_fake_scale,
// mp_fake_store): what the codes and scale of rowquant_kernel / moe_permute_quant_kernel multiply to, bit for
// bit.  One workgroup per row, the row in registers (V 16-byte chunks per thread; V = 0: any K and
// alignment, two passes).  With row_of_slot, workgroup a writes token a / top_k to routed row
// row_of_slot[a] (negative: none); without, row a in place or elsewhere (a thread reads what it writes).
template <int DT, int V>
__global__ __launch_bounds__(256) void fake_values_kernel(const uint16_t *x, int64_t k, const int32_t *__restrict__ row_of_slot,
                                                          int top_k, uint16_t *y) {
  constexpr int MODE = DT == MP_F16 ? kRoundF16 : kRoundBF16;
  __shared__ float red[3][4];
  __shared__ int wbad[4];
  const int tid = threadIdx.x;
  int64_t src = blockIdx.x, dst = src;
  if (row_of_slot) {
    dst = row_of_slot[src];
    src /= top_k;
    if (dst < 0) return;  // workgroup-uniform
  }
  const uint16_t *xr = x + src * k;
  uint16_t *yr = y + dst * k;
  auto ld = [](uint16_t b) { return DT == MP_F16 ? mp_h2f(b) : mp_bf2f(b); };
  mp_rowstat st{0.f, -INFINITY, INFINITY, 0};
  auto see = [&](float f) {
    st.amax = fmaxf(st.amax, fabsf(f));
    st.vmax = fmaxf(st.vmax, f);
    st.vmin = fminf(st.vmin, f);
  };
  if constexpr (V > 0) {
    uint4 v[V];
    const int64_t nch = k / 8;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int64_t c = tid + 256 * i;
      v[i] = c < nch ? reinterpret_cast<const uint4 *>(xr)[c] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
      if (tid + 256 * i >= nch) continue;
      float f[8];
      mp_chunk_to_f32<DT>(v[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) see(f[e]);
    }
    st = mp_block_rowstat(st, red, wbad);
    float s, sg;
    mp_row_scale<MP_SCALE_FAKE>(st, MODE, 0.f, s, sg);
    const float ss = sg * s;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int64_t c = tid + 256 * i;
      if (c >= nch) continue;
      float f[8];
      mp_chunk_to_f32<DT>(v[i], f);
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = wide_pack2<DT>(static_cast<float>(mp_fake_store(f[2 * e], s, sg, MODE)) * ss,
                              static_cast<float>(mp_fake_store(f[2 * e + 1], s, sg, MODE)) * ss);
      reinterpret_cast<uint4 *>(yr)[c] = make_uint4(o[0], o[1], o[2], o[3]);
    }
  } else {
    for (int64_t c = tid; c < k; c += 256) see(ld(xr[c]));
    st = mp_block_rowstat(st, red, wbad);
    float s, sg;
    mp_row_scale<MP_SCALE_FAKE>(st, MODE, 0.f, s, sg);
    const float ss = sg * s;
    for (int64_t c = tid; c < k; c += 256) {
      const float v = static_cast<float>(mp_fake_store(ld(xr[c]), s, sg, MODE)) * ss;
      yr[c] = DT == MP_F16 ? mp_f2h(v) : mp_f2bf(v);
    }
  }
}

template <int DT>
void fake_values_launch(const uint16_t *x, int64_t rows, int64_t k, const int32_t *row_of_slot, int top_k, uint16_t *y,
                        hipStream_t s) {
  const dim3 g(static_cast<unsigned>(rows));
  const int64_t per = k % 8 == 0 && mp_aligned(x, 16) && mp_aligned(y, 16) ? mp_cdiv(k / 8, 256) : 0;
#define MP_FV(V_) hipLaunchKernelGGL((fake_values_kernel<DT, V_>), g, dim3(256), 0, s, x, k, row_of_slot, top_k, y)
  if (per == 0 || per > 16) MP_FV(0);
  else if (per == 1) MP_FV(1);
  else if (per == 2) MP_FV(2);
  else if (per <= 4) MP_FV(4);
  else if (per <= 8) MP_FV(8);
  else MP_FV(16);
#undef MP_FV
}

}  // namespace

int mp_launch_fake_values(const void *x, int dt, int64_t rows, int64_t k, const int32_t *row_of_slot, int top_k, void *y,
                          hipStream_t stream) {
  if (dt != MP_F16 && dt != MP_BF16) return MP_ERR_DTYPE;
  if (rows > INT32_MAX || k <= 0) return MP_ERR_SHAPE;
  if (rows <= 0) return MP_OK;
  const auto *xp = static_cast<const uint16_t *>(x);
  auto *yp = static_cast<uint16_t *>(y);
  if (dt == MP_F16) fake_values_launch<MP_F16>(xp, rows, k, row_of_slot, top_k, yp, stream);
  else fake_values_launch<MP_BF16>(xp, rows, k, row_of_slot, top_k, yp, stream);
  MP_CHECK_LAUNCH();
  return MP_OK;
}

bool mp_dq_wide_takes(const mp_dq_args &p, int epi) {
  const int64_t nb_rows = epi == MP_EPI_SWIGLU ? 2 * p.n : p.n;
  return p.a_fmt == MP_DQ_DT && p.b_fmt == MP_DQ_I8ROW && (epi == MP_EPI_DENSE || epi == MP_EPI_SWIGLU) &&
         p.k % kWBK == 0 && p.k <= (1 << 20) && nb_rows * p.k < (int64_t(1) << 31) && mp_aligned(p.a, 16) &&
         mp_aligned(p.b, 16) && p.n < (1 << 28) && p.rows < (int64_t(1) << 31) &&
         (epi != MP_EPI_SWIGLU || (p.out_dtype == p.dt && p.n % 8 == 0 && p.ldy % 8 == 0 && mp_aligned(p.y, 16)));
}

int mp_launch_dq_wide(const mp_dq_args &p, int epi, hipStream_t stream) {
  // a few rows of a dense call: measured against the tiled kernel, whole module calls at K = 4096, N = 11008, M = 1 / 8 /
  // 32 26-28 (host-bound; kernel 12.6 us) against 34-35 us, M = 16 at 8192 x 8192 29 against 60 us
  if (epi == MP_EPI_DENSE && !p.offsets && p.rows <= 32 && p.k % 128 == 0 && p.k >= 512) {
    if (p.dt == MP_F16) return p.rows <= 16 ? skinny_launch<MP_F16, 1>(p, stream) : skinny_launch<MP_F16, 2>(p, stream);
    return p.rows <= 16 ? skinny_launch<MP_BF16, 1>(p, stream) : skinny_launch<MP_BF16, 2>(p, stream);
  }
  if (p.dt == MP_F16)
    return epi == MP_EPI_SWIGLU ? wide_pick<MP_F16, MP_EPI_SWIGLU>(p, stream) : wide_pick<MP_F16, MP_EPI_DENSE>(p, stream);
  return epi == MP_EPI_SWIGLU ? wide_pick<MP_BF16, MP_EPI_SWIGLU>(p, stream) : wide_pick<MP_BF16, MP_EPI_DENSE>(p, stream);
}

// SmoothQuantLinear's fake path in one call: the per-token fake-quantized activations into the workspace, then
// the linear on them and on r(q * s) of the weight rows.
static int64_t mp_linear_fake_values(int64_t m, int64_t k) { return mp_cdiv(m * k * 2, 256) * 256; }
// K splits of the linear: where the tiles leave CUs idle and the rows are past the few-row kernel's.
static int mp_linear_fake_splits(int64_t m, int64_t n, int64_t k) {
  return m > 32 && m < 1024 && k % 128 == 0 ? wide_splits(m, n, k) : 1;
}

extern "C" size_t mp_w8a8_linear_fake_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const int s = mp_linear_fake_splits(m, n, k);
  return static_cast<size_t>(mp_linear_fake_values(m, k)) + (s > 1 ? static_cast<size_t>(s) * m * n * 4 : 0);
}

extern "C" int mp_w8a8_linear_fake(const void *x, int dtype, int64_t m, int64_t k, const int8_t *w, const float *s_ch,
                                   int64_t n, const void *bias, void *y, void *workspace, size_t workspace_bytes,
                                   mp_stream_t stream) {
  if (!x || !w || !s_ch || !y) return MP_ERR_ARG;
  if (dtype != MP_F16 && dtype != MP_BF16) return MP_ERR_DTYPE;
  if (m < 0 || n <= 0 || k <= 0) return MP_ERR_SHAPE;
  if (m == 0) return MP_OK;
  if (!workspace || workspace_bytes < mp_w8a8_linear_fake_workspace_bytes(m, n, k)) return MP_ERR_WORKSPACE;
  if (!mp_aligned(workspace, 16)) return MP_ERR_ALIGN;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int rc = mp_launch_fake_values(x, dtype, m, k, nullptr, 1, workspace, s);
  if (rc != MP_OK) return rc;
  const int splits = mp_linear_fake_splits(m, n, k);
  if (splits > 1) {
    mp_dq_args d{};
    d.dt = dtype;
    d.a = workspace;
    d.a_fmt = MP_DQ_DT;
    d.b = w;
    d.b_fmt = MP_DQ_I8ROW;
    d.b_scale = s_ch;
    d.bias = bias;
    d.bias_dtype = dtype;
    d.y = y;
    d.out_dtype = dtype;
    d.ldy = n;
    d.rows = m;
    d.n = n;
    d.k = k;
    float *part = reinterpret_cast<float *>(static_cast<char *>(workspace) + mp_linear_fake_values(m, k));
    if (mp_dq_wide_takes(d, MP_EPI_DENSE))
      return dtype == MP_F16 ? wide_launch<MP_F16, MP_EPI_DENSE, 1>(d, splits, part, s)
                             : wide_launch<MP_BF16, MP_EPI_DENSE, 1>(d, splits, part, s);
  }
  // row parts the descriptors of every kernel of mp_dq_linear reach
  const int64_t part = mp_cdiv(int64_t(1) << 30, k) > 1 ? mp_cdiv(int64_t(1) << 30, k) - 1 : 1;
  for (int64_t r = 0; r < m; r += part) {
    const int rc2 = mp_dq_linear(static_cast<const uint16_t *>(workspace) + r * k, nullptr, w, s_ch, bias, dtype,
                                 static_cast<uint16_t *>(y) + r * n, m - r < part ? m - r : part, n, k, stream);
    if (rc2 != MP_OK) return rc2;
  }
  return MP_OK;
}
