// The direct-to-LDS dequantising GEMM (dqwide.hip) for 16-bit activations and int8 weight rows.
#pragma once
#include <type_traits>

#include "dq_gemm.h"

// Whether the kernel takes these operands (formats, K % 64 == 0, 16-byte aligned A and B, an expert's
// weight rows below 2 GiB; SwiGLU: 16-bit h in the dtype, I % 8 == 0).
bool mp_dq_wide_takes(const mp_dq_args &args, int epilogue);
int mp_launch_dq_wide(const mp_dq_args &args, int epilogue, hipStream_t stream);

// Rows of the per-token fake rule's values r(q * s) in the dtype (see fake_values_kernel); x == y is allowed
// without row_of_slot.
int mp_launch_fake_values(const void *x, int dt, int64_t rows, int64_t k, const int32_t *row_of_slot, int top_k, void *y,
                          hipStream_t stream);
