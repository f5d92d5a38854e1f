// The direct-to-LDS int8 GEMM (i8wide.hip), dense (from 33 rows to thousands) and grouped by expert.
#pragma once
#include "i8_gemm.h"

// Whether the kernel takes the operands: K % 128 == 0, 16-byte aligned A and B, an expert's weights below 2 GiB.
bool mp_i8_wide_takes(const mp_i8_args &args, int epilogue);
int mp_launch_i8_wide(const mp_i8_args &args, int epilogue, hipStream_t stream);

// Dense with K split over workgroups: int32 partials [splits, M, N] (16-byte aligned) and a second launch
// that adds them, exactly, and applies the epilogue.  mp_i8_wide_splits: the splits that give a tile to
// every CU (1: no use).
int mp_i8_wide_splits(int64_t m, int64_t n, int64_t k);
int mp_launch_i8_split(const mp_i8_args &args, int splits, int *partials, hipStream_t stream);
