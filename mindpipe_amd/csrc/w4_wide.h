// The direct-to-LDS W4A16 GEMM (w4wide.hip) for more than a few rows.
#pragma once
#include "mp_common.h"

struct mp_w4_wide_args {
  const uint16_t *x;       // [M, K] in dt
  const uint32_t *w;       // [N, K / 8]
  const uint16_t *scales;  // [N, K / 128] in dt
  const uint16_t *zeros;   // [N, K / 128] in dt, or null (zero point 8)
  const uint16_t *bias;    // [N] in dt, or null
  uint16_t *y;             // [M, N] in dt (SwiGLU: [M, N / 2])
  int dt;                  // MP_F16 / MP_BF16
  int64_t m, n, k;
};

// Whether the kernel takes these operands (group 128 assumed): K % 256 == 0, 16-byte aligned x and w,
// 4-byte aligned scales and zeros, and buffers its 32-bit offsets reach.
bool mp_w4_wide_takes(const mp_w4_wide_args &a, bool swiglu);
// rounded: weights rounded to fp16 as the prefill kernel does (bf16 always rounds); else the group scale is
// applied to the fp32 sum of a group, as the batched fp16 kernel does (not with swiglu).  partials (fp32
// [splits, M, N], 16-byte aligned; not with swiglu) or null: K split over workgroups and a second launch.
int mp_launch_w4_wide(const mp_w4_wide_args &a, bool swiglu, bool rounded, int splits, float *partials, hipStream_t stream);
// Whether the kernel is the faster one without a workspace (group 128).
bool mp_w4_wide_rule(const mp_w4_wide_args &a, bool swiglu);
// Whether the batched kernel's numerics apply to m rows of an n-column fp16 output (w4a16.hip).
bool mp_w4_batch_numerics(int64_t m, int64_t n);
