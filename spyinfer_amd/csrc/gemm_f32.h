// The float32 products (gemm_f32.hip): C[M, N] = A[M, K] . W[N, K]^T, all three float32, rows dense, K a multiple of 4 and both
// operands 16-byte aligned.  gemm_f32_takes: whether they stand for these operands.
#pragma once
#include "common.h"

bool gemm_f32_takes(const void* A, const void* W, const void* C, int M, int N, int K);
int gemm_f32(const float* A, const float* W, float* C, int M, int N, int K, hipStream_t st);

// Many rows (gemm_f32_split.hip): whether its kernel takes the product in `parts` parts of K, C [parts][M][N]; the product; and the one of
// W = [gate rows | up rows] with its activation, C [M][N / 2].  Operands as gemm_f32_takes has them.
bool gemm_f32_split_takes(int M, int N, int K, int parts);
int gemm_f32_split(const float* A, const float* W, float* C, int M, int N, int K, int parts, hipStream_t st);
int gemm_f32_split_gated(const float* A, const float* W, float* C, int M, int N, int K, GateAct act, hipStream_t st);
