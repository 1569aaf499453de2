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

// The results of a block through an LDS stage of STAGE row tiles (16 x 128 bfloat16 each), as many row tiles at a time as fit, in a part that a wave has to
// itself (a wave's LDS accesses stay in order): the sums go there as they are, and a loop of few instructions reads whole pieces of
// rows, forms the values and stores them.  Formed where the sums lie, the values of eight to sixteen row tiles are 10 to 40 KB of instructions that every
// block runs through once, and waits for; and a store from there writes sixteen pieces of 32 bytes (blocks of up to eight row tiles, us, before /
// now: stored 4096 x 2048, 1356 rows 28.0 / 26.9, parts 2560 x 9728, 200 rows 17.8 / 16.3, 409 rows 25.4 / 24.0; experts' down products, 147 KB
// of code before, with the gated ones 32 of 2 x 1536 x 2048, 251 rows each 238 / 233).  A piece of four columns lies at place p ^ (row % 16).
// PAIRED: the wave's columns 32 on are the up values of the first 32.  form(row, v, u): a piece's values in v (their up values in u) become
// results; place(row): the output row of row `row` of the block, or -1; out, ld: the output and its rows' length; at: this wave's first column.
template <int MT, int STAGE, bool PAIRED, typename T, typename ACC, typename F, typename P>
__device__ __forceinline__ void gr_results(ACC (&acc)[4][MT], bf16_t* stage, T* out, int64_t ld, int width, int at, int lane, int wave, F form, P place) {
    constexpr int CT = STAGE / 4, VEC = 16 / sizeof(T), PIECES = (PAIRED ? 32 : 64) / VEC, ROWS = 64 / PIECES;
    static_assert(CT >= 1, "a row tile of four waves fits the stage");
    float* mine = reinterpret_cast<float*>(stage) + wave * CT * 16 * 64;
    const int r = lane & 15, g = lane >> 4, q = (lane % PIECES) * (VEC / 4);
#pragma unroll
    for (int i0 = 0; i0 < MT; i0 += CT) {
#pragma unroll
        for (int i = i0; i < i0 + CT && i < MT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<gr_f32x4_t*>(mine + ((i - i0) * 16 + r) * 64 + ((j * 4 + g) ^ r) * 4) = __builtin_bit_cast(gr_f32x4_t, acc[j][i]);
        __builtin_amdgcn_sched_barrier(0);
        const int rows = 16 * min(CT, MT - i0);
#pragma unroll 1
        for (int row = lane / PIECES; row < rows; row += ROWS) {
            const float* from = mine + row * 64;
            float v[VEC], u[VEC];
#pragma unroll
            for (int k = 0; k < VEC / 4; ++k) {
                const gr_f32x4_t a = *reinterpret_cast<const gr_f32x4_t*>(from + ((q + k) ^ (row & 15)) * 4);
                const gr_f32x4_t b = PAIRED ? *reinterpret_cast<const gr_f32x4_t*>(from + ((q + k + 8) ^ (row & 15)) * 4) : a;
#pragma unroll
                for (int e = 0; e < 4; ++e) { v[k * 4 + e] = a[e]; u[k * 4 + e] = b[e]; }
            }
            const int64_t to = place(i0 * 16 + row);
            form(i0 * 16 + row, v, u);
            if (to >= 0 && at + q * 4 < width) {
                T* o = out + to * ld + at + q * 4;
                if constexpr (sizeof(T) == 2) *reinterpret_cast<uint4*>(o) = uint4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
                else *reinterpret_cast<gr_f32x4_t*>(o) = gr_f32x4_t{v[0], v[1], v[2], v[3]};
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// What a block of 16 MT rows from row0 on and 256 rows of W writes (gemm_rows.hip has what is formed).
template <int MT, int STAGE, int EPI, typename ACC>
__device__ __forceinline__ void gr_block_out(ACC (&acc)[4][MT], bf16_t* stage, void* C, int M, int N, int row0, int col_t, int part, const GateAct& act, int lane, int wave) {
    const auto row_of = [](int row) { return (int64_t)row; };
    if constexpr (EPI == ROWS_PARTS) {
        gr_results<MT, STAGE, false>(acc, stage, (float*)C + ((size_t)part * M + row0) * N, N, N, col_t * 256 + wave * 64, lane, wave, [](int, float (&)[4], float (&)[4]) {}, row_of);
    } else if constexpr (EPI == ROWS_STORE) {
        gr_results<MT, STAGE, false>(acc, stage, (bf16_t*)C + (size_t)row0 * N, N, N, col_t * 256 + wave * 64, lane, wave, [](int, float (&)[8], float (&)[8]) {}, row_of);
    } else {
        gr_results<MT, STAGE, true>(acc, stage, (bf16_t*)C + (size_t)row0 * (N / 2), N / 2, N / 2, col_t * 128 + wave * 32, lane, wave, [&](int, float (&v)[8], float (&u)[8]) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = gated_value_short(act, v[e], u[e]);
        }, row_of);
    }
}
