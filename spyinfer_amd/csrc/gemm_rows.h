// What the products of many bfloat16 rows share: what is formed, the operand types, the arguments of a launch.
#pragma once
#include "common.h"

#define ROWS_STORE 0
#define ROWS_PARTS 1
#define ROWS_GATED 2
#define ROWS_DIES 8

typedef __bf16 gr_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float gr_f32x4_t __attribute__((ext_vector_type(4)));

// Blocks of nine row tiles and more, one a compute unit (gemm_rows_tall.hip); n_rows blocks share a column's rows, MT row tiles each.
int gr_tall_launch(void* C, const void* X, const void* W, int M, int N, int K, int MT, int n_rows, int parts, int epi, GateAct act, hipStream_t st);
