// Products of many bfloat16 rows (prompts, portions of prompts) from the matrix' tiled copy (gemm_decode.h has the order), float32
// sums on v_mfma_f32_16x16x32_bf16:
//   ROWS_PARTS:  K cut into parts, one block each: parts[p][M][N] float32, added in the pass of the norm that reads the result
//                (spy_add_parts_rmsnorm), which reads the stream there anyway;
//   ROWS_STORE:  C[M][N] in bfloat16;
//   ROWS_GATED:  W = [gate rows | up rows], C[M][N / 2] = act(gate) * up in bfloat16, without the [M][N] tensor in between.
//
// A block has 16 MT rows of X and 256 rows of W (gated: 128 gate rows and the 128 up rows of the same columns); each of its four
// waves has all of the rows and 64 of W's, so W goes from memory straight into MFMA operand registers (1 KB a load, every byte
// loaded by one wave) and LDS carries X alone: 64 bytes a clock and compute unit where 2 x 2 waves with both operands in LDS need
// 128, all there is.  A turn is 128 of K: X's next 128 go from memory into the other of two LDS stages while this one's 16 MT
// products run, and a step's W registers are asked for again, for the next turn, as soon as their last product is issued.  Piece p of
// an LDS row lies at place p ^ (row % 16), which the lanes' source addresses see to, so that the operands' reads meet in no bank.
// Two blocks fit a compute unit.  (Blocks of 9 to 16 row tiles, one a unit: gemm_rows_tall.hip; which of the two: rows_product_tall in kernels/ops.py.)  Turns of 256 (twice the bytes under way) and loads spread over the products one by one were not faster.
//
// Why parts: a prompt of a few hundred rows has fewer tiles than compute units, and each would walk all of K alone.  Measured (us;
// library, this kernel, and what the sum of its parts adds to the norm's pass):  409 rows, 2560 x 9728: 53.7, 27.8 + 5 (six parts);
// 2560 x 4096: 23.8, 17.2 + 4; 200 rows, 4096 x 12288: 50.7, 31.2 + 6; 800 rows, 2048 x 6144: 39.0, 28.4 + 4.  Gated, with the
// library's activation pass: 409 rows, 19456 x 2560: 53.2 + 8, 57.7; 1356 rows, 12288 x 2048: 85.6 + 13, 70.7 (965 TFLOP/s); 130 rows,
// 19456 x 2560: 40.8 + 5, 33.2.
// (Each with expf and a division in the epilogue; with gated_value_short 409 rows 46.1 -> 45.1, 1356 rows 65.4 -> 63.5, 2048 rows, 24576 x 4096 333 -> 323.)
// What bounds it: a turn takes 0.7 + 0.05 MT us, its 16 MT products per SIMD 0.11 MT us of that at four waves a compute unit; the rest
// is the loads' way, from memory where few tiles share W, and the turn's barrier.
#include "gemm_rows.h"

// X and W are not declared free of aliases: the waits below count the loads issued before them, and with that promise the compiler may
// move loads of W across a wait.  STAGE: row tiles that an LDS stage has room for.
template <int MT, int STAGE, int EPI>
__device__ __forceinline__ void gemm_rows_block(void* C, const bf16_t* X, const bf16_t* W, int M, int N, int K, int col_t, int part, int parts, int tile0,
                                                GateAct act, bf16_t* stage0, bf16_t* stage1) {
    const int chunks = K / 128, c0 = (int)((long long)chunks * part / parts);
    const int n = (int)((long long)chunks * (part + 1) / parts) - c0;                  // (at least one: the launcher's check)
    // The last rows' tile ends with row M - 1 (M >= 16 MT): what it shares with the tile before, both blocks form alike
    const int row0 = min(tile0 * 16, M - MT * 16);
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NT = N / 16;
    // byte offsets below 2^31 (the launcher's check)
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
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = gr_f32x4_t{0.f, 0.f, 0.f, 0.f};
    gr_bf16x8_t w[4][4];
    auto load_x = [&](bf16_t* stage, int c) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (__attribute__((address_space(3))) void*)(stage + (i * 4 + wave) * 512), 16, x_lane,
                                                     x_at + i * 32 * K + c * 256, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_w = [&](int s, int c) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[s][j] = __builtin_bit_cast(gr_bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(wres, w_lane, w_at[j] + c * w_turn + s * 1024, 0));
    };
    // the products of one turn; `next`: the turn whose W is asked for (none if negative).  X's operands are read three ahead.
    auto products = [&](const bf16_t* stage, int next, bool more) {
        const bf16_t* xb = stage + r * 128;
        gr_bf16x8_t x[4];
#pragma unroll
        for (int q = 0; q < 3; ++q) x[q] = *reinterpret_cast<const gr_bf16x8_t*>(xb + (q % MT) * 2048 + ((4 * (q / MT) + g) ^ r) * 8);
#pragma unroll
        for (int q = 0; q < 4 * MT; ++q) {
            const int s = q / MT, i = q % MT, ahead = q + 3;
            if (ahead < 4 * MT) x[ahead % 4] = *reinterpret_cast<const gr_bf16x8_t*>(xb + (ahead % MT) * 2048 + ((4 * (ahead / MT) + g) ^ r) * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][j], x[q % 4], acc[j][i], 0, 0, 0);
            if (i == MT - 1 && more) load_w(s, next);
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
    load_x(stage0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) load_w(s, 0);
    turn();
    // (two turns a round, whatever is left: loads that a branch skips would make the compiler count fewer under way.  The last round
    // asks for the last turn once more; its own tail loop costs 130 to 390 registers spilled at six to eight row tiles)
    int c = 0;
    for (; c + 1 < n; c += 2) {
        load_x(stage1, c + 1);
        products(stage0, c + 1, true);
        turn();
        const int after = min(c + 2, n - 1);
        load_x(stage0, after);
        products(stage1, after, true);
        turn();
    }
    if (c < n) products(stage0, 0, false);
    if (EPI == ROWS_GATED) {
        // (formed where the sums lie: behind LDS, as the other results, 500 rows, 6144 x 1024 take 11.2 us for 10.6, 640 rows, 12288 x 2048 32.4 for 31.7)
        const int NG = NT / 2;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            bf16_t* c_row = (bf16_t*)C + (size_t)(row0 + i * 16 + r) * (N / 2) + 4 * g;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int tile = col_t * 8 + wave * 2 + j;
                float y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = gated_value_short(act, acc[j][i][e], acc[j + 2][i][e]);
                const uint2 o = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
                if (tile < NG) *reinterpret_cast<uint2*>(c_row + tile * 16) = o;
            }
        }
        return;
    }
    // (nothing under way into the stages, and nobody reads them)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EPI != ROWS_GATED) gr_block_out<MT, STAGE, EPI>(acc, stage0, C, M, N, row0, col_t, part, act, lane, wave);
}

// A column of tiles (256 columns, one part) has n_rows blocks, `tall` of them with MT row tiles and the others with one less, as many in
// all as the rows need.  Which ones are tall moves on by `tall` from one column to the next, so that those that follow each other on a
// compute unit are of both kinds.  Where all are tall nothing of that is worked out, and up to five row tiles the kernel has no code for the other
// size either (DEALT false); more tiles are scheduled worse without it.  Stored, us, dealt / tall in the same kernel / without: 80 rows, 4096 x 1024
// 11.15 / 11.06 / 10.68, 640 rows 12.19 / 12.14 / 11.70, 200 rows 11.02 / 10.80 / 10.98, 1700 rows 20.95 / 20.29 / 20.85.
template <int MT, int EPI, bool DEALT>
__global__ __launch_bounds__(256, 2) void gemm_rows_kernel(void* C, const bf16_t* X, const bf16_t* W, int M, int N, int K, int n_rows, int tall,
                                                           int n_cols, int parts, int blocks, GateAct act) {
    __shared__ __align__(1024) bf16_t stage0[MT * 16 * 128];
    __shared__ __align__(1024) bf16_t stage1[MT * 16 * 128];
    // Blocks go to the dies in turn: a die takes a run of the blocks in (part, columns, rows) order, so that the blocks that read the
    // same rows of W run beside each other and the matrix comes into one L2 once
    const int per = (blocks + ROWS_DIES - 1) / ROWS_DIES, idx = blockIdx.x / ROWS_DIES;
    const int v = (blockIdx.x % ROWS_DIES) * per + idx;
    if (idx >= per || v >= blocks) return;
    const int cp = v / n_rows, i = v % n_rows, col_t = cp % n_cols, part = cp / n_cols;
    if (!DEALT || tall == n_rows) {
        gemm_rows_block<MT, MT, EPI>(C, X, W, M, N, K, col_t, part, parts, i * MT, act, stage0, stage1);
        return;
    }
    const int shift = (int)((unsigned)cp * (unsigned)tall % (unsigned)n_rows), at = i + shift;
    const int before = (at >= n_rows ? tall + min(at - n_rows, tall) : min(at, tall)) - min(shift, tall);      // tall blocks before this one
    const int tile0 = i * (MT - 1) + before;
    if ((at >= n_rows ? at - n_rows : at) < tall) gemm_rows_block<MT, MT, EPI>(C, X, W, M, N, K, col_t, part, parts, tile0, act, stage0, stage1);
    else gemm_rows_block<MT - 1, MT, EPI>(C, X, W, M, N, K, col_t, part, parts, tile0, act, stage0, stage1);
}

template <int MT>
static int rows_launch(void* C, const void* X, const void* W, int M, int N, int K, int n_rows, int parts, int epi, GateAct act, hipStream_t st) {
    // (blocks of four tiles overlap where there are not four for each)
    const int n_cols = (N + 255) / 256, left = (M + 15) / 16 - n_rows * (MT - 1), tall = MT == 4 && left < 1 ? n_rows : left;
    const int64_t blocks = (int64_t)n_rows * n_cols * parts;
    SPY_REQUIRE(M >= MT * 16 && tall >= 1 && tall <= n_rows && blocks < (1 << 30), "spy_gemm_rows: %d rows in %d tiles of %d, %lld blocks", M, n_rows, MT, (long long)blocks);
    const unsigned grid = (unsigned)((blocks + ROWS_DIES - 1) / ROWS_DIES * ROWS_DIES);
#define ROWS_N(EPI, PARTS, DEALT) gemm_rows_kernel<MT, EPI, DEALT><<<grid, 256, 0, st>>>(C, (const bf16_t*)X, (const bf16_t*)W, M, N, K, n_rows, tall, n_cols, PARTS, (int)blocks, act)
#define ROWS(EPI, PARTS) do { if (MT <= 5 && tall == n_rows) ROWS_N(EPI, PARTS, (MT > 5)); else ROWS_N(EPI, PARTS, true); } while (0)
    if (epi == ROWS_STORE) ROWS(ROWS_STORE, 1);
    else if (epi == ROWS_GATED) ROWS(ROWS_GATED, 1);
    else ROWS(ROWS_PARTS, parts);
#undef ROWS
#undef ROWS_N
    SPY_CHECK_LAUNCH("spy_gemm_rows");
    return 0;
}

// Blocks that share a column's rows, of at most `most` row tiles each.  A compute unit's time is the row tiles of its blocks together, whether
// they run beside or behind each other (1356 rows, 12288 x 2048: 720 blocks of six, three a unit, 65 us; 816 of five, four a unit, 72; 624 of
// seven, three a unit, 70), so where it has two or more, as many blocks as leave its number of them what it is, and the rows dealt
// evenly to them (409 rows, 19456 x 2560, six blocks of five and four 50.3 us, of five 51.4; 640 rows, six of seven and six 58.1 / 59.5).  With one a
// unit the largest counts, and the fewest blocks stand.
static int rows_blocks(int tiles, int most, int columns) {
    const int fewest = (tiles + most - 1) / most, each = (int)(((int64_t)fewest * columns + 255) / 256);
    if (each < 2) return fewest;
    return max(fewest, (int)min((int64_t)256 * each / columns, (int64_t)tiles / 4));
}

// epi: what is formed (see the top): C bfloat16 [M, N], float32 [parts, M, N] or bfloat16 [M, N / 2].  X: bfloat16 rows [M, K]; W: the tiled copy of [N, K].  row_tiles: most of a block, 4 to 16.
extern "C" int spy_gemm_rows(void* C, const void* X, const void* W, int M, int N, int K, int row_tiles, int parts, int epi, int act_code,
                             hipStream_t st) {
    GateAct act = {1.f, 0.f};
    SPY_REQUIRE(M > 0 && N > 0 && K > 0 && N % (epi == ROWS_GATED ? 32 : 16) == 0 && K % 128 == 0, "spy_gemm_rows: bad sizes %d x %d x %d", M, N, K);
    SPY_REQUIRE((int64_t)N * K < (1 << 30) && (int64_t)M * K < (1 << 30), "spy_gemm_rows: operands of %d x %d x %d are too large", M, N, K);
    SPY_REQUIRE(parts >= 1 && parts <= K / 128 && (parts == 1 || epi == ROWS_PARTS) && epi >= ROWS_STORE && epi <= ROWS_GATED, "spy_gemm_rows: %d parts of K = %d", parts, K);
    SPY_REQUIRE((((uintptr_t)C | (uintptr_t)X | (uintptr_t)W) % 16) == 0, "spy_gemm_rows: operands must be 16-byte aligned");
    SPY_REQUIRE(epi != ROWS_GATED || gate_act_of(act_code, &act), "spy_gemm_rows: unknown activation %d", act_code);
    SPY_REQUIRE(row_tiles >= 4 && row_tiles <= 16, "spy_gemm_rows: %d row tiles", row_tiles);
    const int tiles = (M + 15) / 16;
    if (row_tiles > 8) {
        const int shared = (tiles + row_tiles - 1) / row_tiles, MT = (tiles + shared - 1) / shared;
        SPY_REQUIRE(MT > 8, "spy_gemm_rows: %d rows make no blocks of %d row tiles", M, row_tiles);
        return gr_tall_launch(C, X, W, M, N, K, MT, shared, parts, epi, act, st);
    }
    const int n_rows = rows_blocks(tiles, row_tiles, (N + 255) / 256 * parts);
    switch (max(4, (tiles + n_rows - 1) / n_rows)) {
        case 4: return rows_launch<4>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 5: return rows_launch<5>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 6: return rows_launch<6>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 7: return rows_launch<7>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
        case 8: return rows_launch<8>(C, X, W, M, N, K, n_rows, parts, epi, act, st);
    }
    return spy_fail("spy_gemm_rows: %d row tiles", row_tiles);
}
