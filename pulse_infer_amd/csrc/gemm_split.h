// The float32 product on the bfloat16 matrix instruction (gemm_split.hip), for gemm_f32's entry points.
#pragma once
#include "common.h"

// Whether products with weights of N rows of K values are made this way.
bool pulse_split_takes(int N, int K);

// How many bytes of scratch the fastest way for these sizes takes (0: none).
int64_t pulse_split_scratch(int M, int N, int K);

// Operands that are read four values at a time; `scratch` null: a way that takes none.
void pulse_split_launch(const float* A, const float* W, void* C, bool c_bf16, bool c_wide, int M, int N, int K, int64_t lda, int64_t ldw,
                        int64_t ldc, void* scratch, hipStream_t stream);
