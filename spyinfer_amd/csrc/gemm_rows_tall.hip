// Products of many bfloat16 rows by blocks of 9 to 16 row tiles of X and 256 rows of W, one block a compute unit and one wave a SIMD
// (gemm_rows.hip has what is formed, the operands' order and the blocks of up to eight row tiles, two a unit).
//
// As there, each of a block's four waves has all rows and 64 of W's, W goes from memory straight into operand registers, X through two LDS
// stages, a turn is 128 of K.  A lone wave has nobody to fill its gaps, so:
//   - the sums are held in accumulation registers by the instructions' own form: given the choice, the compiler keeps some of them
//     and of W on the wrong side and moves 100 to 200 registers a turn;
//   - W is asked for a turn and more ahead (two turns of it in registers), which covers its way from memory;
//   - loads are issued one by one between the products.  Four waves' loads of a kilobyte each take the address unit 64 clocks, so
//     bursts of 4 and of MT at a turn's ends held the products up: a turn of nine row tiles took 3400 clocks, spread 2850, its
//     products alone 2304; of thirteen 3780 of 3328;
//   - results leave through LDS, so that a store's lanes write whole lines of a row (6144 x 4096, 2048 rows: 81 -> 73 us; straight from the
//     sums a store is sixteen pieces of 32 bytes, and thirteen row tiles' took 14 250 clocks), formed by a short loop on their way
//     (24576 x 4096 gated, 2048 rows: 292 -> 287 us).
// A turn's X and W are 64 KB + 4 KB a row tile, so a product of thirteen row tiles moves 45 KB for what one of five moves 84 KB: the first-level
// caches and L2s, which the small blocks keep busy, have half the work.  Measured, us, the small blocks or the library (with its activation's
// pass, with the norm that sums parts) / this: gated, 19456 x 2560, 409 rows 53.5 / 41.6 (0.98 PFLOP/s), 24576 x 4096, 300 rows 75.4 / 62.4,
// 2048 rows 302 / 291 (1.42); stored, 6144 x 4096, 2048 rows 83.6 / 75.6 (1.36), 6144 x 2048, 1356 rows 45.1 / 30.7; parts, 4096 x
// 12288, 2048 rows 193 / 169.  Where the line to the small blocks lies: rows_product_tall in kernels/ops.py.
// What bounds it: at thirteen row tiles the matrix units are busy for 88 % of a turn and the clock falls to 1.6 to 1.9 GHz; at nine a turn's loads,
// 26 % over its products, and a block's way in (2.2 us to its first turn) and out (2 to 4 us), which a lone wave a SIMD shows.
#include "gemm_rows.h"

// Two products of a row tile, X's 16 rows with two column tiles of W.  The compiler does not see matrix instructions here and leaves out the
// wait states between them and ordinary instructions: an operand's register that one has written needs two (a turn begins with them, and
// inside of it there are none: tests/test_rows_tall_listing.py looks), and what reads the sums waits for the last product (gr_sums_settle).
// Two before every pair cost 3 to 9 %.
__device__ __forceinline__ void gr_mfma2(gr_f32x4_t& a, gr_f32x4_t& b, gr_bf16x8_t w0, gr_bf16x8_t w1, gr_bf16x8_t x) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %2, %4, %0\n\tv_mfma_f32_16x16x32_bf16 %1, %3, %4, %1" : "+a"(a), "+a"(b) : "v"(w0), "v"(w1), "v"(x));
}
__device__ __forceinline__ void gr_sums_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// All turns of a block: n of them, of 128 of K.  wres, w_lane, w_at, w_turn: W's buffer, this lane's bytes in a load, each column tile's place and a
// turn's bytes.  load_x(stage, i, c): asks for row tile i of turn c, straight into LDS (a wave 4 of its 16 rows).  Ends with nothing under way,
// the stages free and the sums fit to be read.  MT: 8 to 16.
template <int MT, typename RES, typename X>
__device__ __forceinline__ void gr_tall_turns(gr_f32x4_t (&acc)[4][MT], RES wres, int w_lane, const int (&w_at)[4], int w_turn, int n, bf16_t* stage0, bf16_t* stage1,
                                              int lane, X load_x) {
    // (two arrays of their own: reads of a stage that the compiler cannot tell from the one that loads go to wait for these)
    static_assert(MT >= 8 && MT <= 16, "eight loads of W go between the row tiles of a step");
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = gr_f32x4_t{0.f, 0.f, 0.f, 0.f};
    gr_bf16x8_t w[2][4][4];
    auto load_w = [&](int d, int s, int j, int c) {
        w[d][s][j] = __builtin_bit_cast(gr_bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(wres, w_lane, w_at[j] + c * w_turn + s * 1024, 0));
    };
    // The products of a turn with w[d].  Between them, one load a row tile: X of turn `next` into the other stage while step 0 runs; W of turn
    // `after` into the registers of steps 0 to 2 as soon as these are done; and, in step 1, W of turn `next` into the other set's
    // step 3, which the turn before had used to its end.  X's operands are read three ahead.
    auto products = [&](int d, const bf16_t* stage, bf16_t* other, int next, int after) {
        const bf16_t* xb = stage + r * 128;
        gr_bf16x8_t x[4];
#pragma unroll
        for (int q = 0; q < 3; ++q) x[q] = *reinterpret_cast<const gr_bf16x8_t*>(xb + (q % MT) * 2048 + ((4 * (q / MT) + g) ^ r) * 8);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 1");
#pragma unroll
        for (int q = 0; q < 4 * MT; ++q) {
            const int s = q / MT, i = q % MT, ahead = q + 3;
            if (ahead < 4 * MT) x[ahead % 4] = *reinterpret_cast<const gr_bf16x8_t*>(xb + (ahead % MT) * 2048 + ((4 * (ahead / MT) + g) ^ r) * 8);
            gr_mfma2(acc[0][i], acc[1][i], w[d][s][0], w[d][s][1], x[q % 4]);
            __builtin_amdgcn_sched_barrier(0);
            if (s == 0) load_x(other, i, next);
            else if (i < 4) load_w(d, s - 1, i, after);
            else if (s == 1 && i < 8) load_w(1 - d, 3, i - 4, next);
            __builtin_amdgcn_sched_barrier(0);
            gr_mfma2(acc[2][i], acc[3][i], w[d][s][2], w[d][s][3], x[q % 4]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // A turn issues X's loads before its 16 loads of W, and loads return in order: at most 16 under way means that X is there
    auto turn = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < MT; ++i) load_x(stage0, i, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) load_w(0, s, j, 0);
    turn();
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) load_w(1, s, j, min(1, n - 1));
    __builtin_amdgcn_sched_barrier(0);
    // (the last turns ask for the last turn's operands again: loads that a branch skips would make the compiler count fewer under way)
    int c = 0;
    for (; c + 1 < n; c += 2) {
        const int after = min(c + 2, n - 1);
        products(0, stage0, stage1, c + 1, after);
        turn();
        products(1, stage1, stage0, after, min(c + 3, n - 1));
        turn();
    }
    if (c < n) products(0, stage0, stage1, n - 1, n - 1);
    gr_sums_settle();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

template <int MT, int EPI>
__global__ __launch_bounds__(256, 1) void gemm_rows_tall_kernel(void* C, const bf16_t* X, const bf16_t* W, int M, int N, int K, int n_rows, int n_cols,
                                                                int parts, int blocks, GateAct act) {
    __shared__ __align__(1024) bf16_t stage0[MT * 16 * 128];
    __shared__ __align__(1024) bf16_t stage1[MT * 16 * 128];
    // (a die takes a run of the blocks in (part, columns, rows) order: see gemm_rows_kernel)
    const int per = (blocks + ROWS_DIES - 1) / ROWS_DIES, idx = blockIdx.x / ROWS_DIES;
    const int v = (blockIdx.x % ROWS_DIES) * per + idx;
    if (idx >= per || v >= blocks) return;
    const int cp = v / n_rows, col_t = cp % n_cols, part = cp / n_cols;
    const int chunks = K / 128, c0 = (int)((long long)chunks * part / parts);
    const int n = (int)((long long)chunks * (part + 1) / parts) - c0;                  // (at least one: the launcher's check)
    const int row0 = min((v % n_rows) * MT * 16, M - MT * 16);                         // the last rows' tile ends with row M - 1
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NT = N / 16;
    const auto wres = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, N * K * 2, 0x00020000);
    const auto xres = __builtin_amdgcn_make_buffer_rsrc((void*)X, 0, M * K * 2, 0x00020000);
    const int w_lane = lane * 16, w_turn = N * 256;
    int w_at[4];                                       // this wave's column tiles; one that does not exist reads the last (nothing is stored)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        int tile;
        if (EPI == ROWS_GATED) tile = (j >> 1) * (NT / 2) + min(col_t * 8 + wave * 2 + (j & 1), NT / 2 - 1);
        else tile = min(col_t * 16 + wave * 4 + j, NT - 1);
        w_at[j] = __builtin_amdgcn_readfirstlane(c0 * w_turn + tile * 4096);
    }
    // X: a wave's load brings 4 rows of 256 bytes; lane l has the piece that belongs to place l % 16 of row l / 16
    const int s_row = wave * 4 + (lane >> 4);
    const int x_lane = (s_row * K + ((lane & 15) ^ s_row) * 8) * 2, x_at = (row0 * K + c0 * 128) * 2;
    gr_f32x4_t acc[4][MT];
    gr_tall_turns<MT>(acc, wres, w_lane, w_at, w_turn, n, stage0, stage1, lane, [&](bf16_t* stage, int i, int c) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (__attribute__((address_space(3))) void*)(stage + (i * 4 + wave) * 512), 16, x_lane,
                                                 x_at + i * 32 * K + c * 256, 0, 0);
    });
    gr_block_out<MT, MT, EPI>(acc, stage0, C, M, N, row0, col_t, part, act, lane, wave);
}

template <int MT>
static int tall_launch(void* C, const void* X, const void* W, int M, int N, int K, int n_rows, int parts, int epi, GateAct act, hipStream_t st) {
    const int n_cols = (N + 255) / 256;
    const int64_t blocks = (int64_t)n_rows * n_cols * parts;
    SPY_REQUIRE(M >= MT * 16 && (int64_t)n_rows * MT * 16 >= M && blocks < (1 << 30), "spy_gemm_rows: %d rows in %d tiles of %d, %lld blocks", M, n_rows, MT, (long long)blocks);
    const unsigned grid = (unsigned)((blocks + ROWS_DIES - 1) / ROWS_DIES * ROWS_DIES);
#define TALL(EPI, PARTS) gemm_rows_tall_kernel<MT, EPI><<<grid, 256, 0, st>>>(C, (const bf16_t*)X, (const bf16_t*)W, M, N, K, n_rows, n_cols, PARTS, (int)blocks, act)
    if (epi == ROWS_STORE) TALL(ROWS_STORE, 1);
    else if (epi == ROWS_GATED) TALL(ROWS_GATED, 1);
    else TALL(ROWS_PARTS, parts);
#undef TALL
    SPY_CHECK_LAUNCH("spy_gemm_rows");
    return 0;
}

int gr_tall_launch(void* C, const void* X, const void* W, int M, int N, int K, int MT, int n_rows, int parts, int epi, GateAct act, hipStream_t st) {
    switch (MT) {
        case 9: return tall_launch<9>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 10: return tall_launch<10>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 11: return tall_launch<11>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 12: return tall_launch<12>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 13: return tall_launch<13>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 14: return tall_launch<14>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 15: return tall_launch<15>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 16: return tall_launch<16>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
    }
    return spy_fail("spy_gemm_rows: %d row tiles", MT);
}
