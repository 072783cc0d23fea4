// The float32 product on the bfloat16 matrix cores (gemm_f32_split.hip).
#pragma once
#include "common.h"

// Whether a float32 weight of K columns takes it: K alone, so that a row's result does not depend
// on the other rows of a call.
inline bool gemm_f32_split_fits(int K) { return K % 64 == 0; }
// float32 operands, 16-byte aligned, and result.  `tile` 0 lets the sizes choose; 1 to 10 name one
// (1 to 3: of 16 rows each at most; the result is the same to the bit).  Returns 0, or -1 where a
// tile needs more LDS than the device gives.
int gemm_f32_split_launch(const float* A, const float* W, float* C, int M, int N, int K, int tile,
                          hipStream_t stream);
