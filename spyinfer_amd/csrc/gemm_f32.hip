// C[M, N] = A[M, K] . W[N, K]^T in float32: products and sums of 32-bit numbers, no reduced-precision mode (the matrix cores'
// float32 instructions multiply and add as fmaf does; gemm_f32_split.hip, which has most products of more than 32 rows, cuts the
// numbers into parts that keep their 24 bits, and leaves those that cannot be cut so to float32 instructions).  Four kernels by the number of rows:
//
//   few    (up to 8 rows)   bound by streaming W from memory: a block's waves share K, 64 lanes side by side along it.
//   narrow (tens of rows)   bound by W from memory as well, but A's rows would be read once per row of W by the kernel above.
//                           A block owns 16 rows of W and MT tiles of 16 rows of A; its eight waves take the chunks of 64 of K in
//                           turn, operands straight from memory into v_mfma_f32_16x16x4_f32 registers, and add through LDS.
//   held   (up to 32 rows of which K is a multiple of 512, up to 2048 or in parts of that)      the same for more tiles of W than compute
//                           units, or for parts of K beside each other: a block stays, its waves keep A in registers.
//   tile   (many rows that gemm_f32_split.hip does not take)      bound by the matrix cores (256 flops a cycle and compute unit).  Tiles of
//                           A and W through LDS.
//
// Which kernel, how many row tiles a block and how many parts of K follow the number of rows, and with them the order of a row's sums: a
// row in a step of other sizes is the same within rounding, not bit for bit (as it is from gemm_generic.hip).
//
// The operands' order of K inside an MFMA step is free as long as both agree: a lane (r = lane % 16, g = lane / 16) loads the four
// values k + 4 g .. + 3 of its row in one piece, and instruction j of four multiplies the j-th of them.
#include "gemm_f32.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gf_f32x4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float gf_f32x16_t;

__device__ __forceinline__ gf_f32x4_t gf_load(const float* p) { return *reinterpret_cast<const gf_f32x4_t*>(p); }
__device__ __forceinline__ gf_f32x4_t gf_stream(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const gf_f32x4_t*>(p)); }

// ---- few rows ------------------------------------------------------------------------------------------------------------
// V sums over each 16 lanes of a wave at once, without LDS: partners are lanes l ^ 15, l ^ 7, l ^ 3, l ^ 1 (moves within a row of lanes), of
// which one keeps the lower half of the values and the other the upper.  Lane l ends with V / 16 sums, of the values from l % 16 V / 16 on
// (V < 16: with one, of value l % 16 / (16 / V)).
template <int CTRL> __device__ __forceinline__ float gf_moved(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL, int BIT, int N, int V>
__device__ __forceinline__ void gf_row_step(float (&v)[V], int lane) {
    if constexpr (N >= 2) {
        const bool upper = (lane & BIT) != 0;
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const float keep = upper ? v[i + N / 2] : v[i], give = upper ? v[i] : v[i + N / 2];
            v[i] = keep + gf_moved<CTRL>(give);
        }
    } else {
        v[0] += gf_moved<CTRL>(v[0]);
    }
}
template <int V>
__device__ __forceinline__ void gf_row_sums(float (&v)[V], int lane) {
    gf_row_step<0x140, 8, V>(v, lane);                                    // row_mirror
    gf_row_step<0x141, 4, (V >= 2 ? V / 2 : 1)>(v, lane);                 // row_half_mirror
    gf_row_step<0x1b, 2, (V >= 4 ? V / 4 : 1)>(v, lane);                  // quad_perm 3 2 1 0
    gf_row_step<0xb1, 1, (V >= 8 ? V / 8 : 1)>(v, lane);                  // quad_perm 1 0 3 2
}

// A block owns NR rows of W; its WV waves take the chunks of 256 of K in turn, U of them and A's pieces asked for at once, and the next
// ones before these are multiplied; the sums of 16 lanes meet in registers, those of a block's rows of lanes in LDS.  Every load of W is 1
// KiB in one piece, and A's rows come out of the caches once per NR rows of W: with a row or two of W a wave, as this kernel had it, A was
// twice to four times W's bytes on a compute unit's way from L2.  Sums over a wave by lane exchanges through LDS took 2.5 us of a launch.
// GATED: W = [gate rows | up rows] of N columns each; a block owns NR / 2 columns, their gate rows and their up rows, and stores act(gate)
// * up.  Measured, us, with one to four rows of W a wave and its own K / this, 4 rows of A: 2048 x 2048 6.9 / 5.6, 2048 x 6144 15.6 / 10.6 (4.7
// TB/s), 4096 x 2048 9.7 / 8.2, 12288 x 2048 gated 22.3 / 18.3 (5.5 TB/s), 151936 x 2048 192 / 186; 1 row: 2048 x 6144 10.3 / 9.9, 1024 x 3072
// 4.1 / 3.95; 8 rows, the narrow kernel / this: 2048 x 6144 23.4 / 13.8, 12288 x 2048 with its activation 45 / 22, 151936 x 2048 356 / 225.
//
// INTO and SCALED fold the norm between two products into them, as gemm_decode.hip does for bfloat16 rows (a norm kernel is 3.7 us between two
// products of 5 to 20; a step of 4 requests, 28 layers 2048 wide, 2064 / 1952 us, the products each as long as before).  INTO: C is the residual stream, which the result is added to; the block also stores the new values times the next
// norm's weight and, for every row, the sum of their squares over its columns (fold.squares [blocks][MR]).  SCALED: A is such a product's
// rows, and the results are scaled by 1 / sqrt(sum / K + eps).  A block reads all of the squares, one for each row (rounded up to 1, 2,
// 4 or 8) of every block of the product that wrote them: for a stream of 2048, 8 KB behind a product of 2048 x 2048 with one row of A, else 2 KB a row, beside
// the 8 KB of a row of A.  What its threads ask for at their start, 2048 squares, is there by the end; beyond, the block waits: the line of
// folded_f32_pays in kernels/ops.py.  (A's rows squared and multiplied by the weight as they come by, without all that, cost the registers of a block or two a
// compute unit: gate/up of 12288 x 2048, 4 rows, 21.2 us for 19.5.)
struct GfFold {
    const float* squares_in;
    int n_squares;             // of squares_in: parts times MR
    float eps;
    float* rows_out;
    const float* weight;
    float* squares_out;
};
template <int CTRL> __device__ __forceinline__ float gf_rotated_sum(float v) { return v + gf_moved<CTRL>(v); }

template <int MR, int NR, int U, int WV, bool GATED, bool SCALED, bool INTO>
__global__ __launch_bounds__(WV * 64) void gemm_f32_few_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                                                              int M, int N, int K, GateAct act, GfFold fold) {
    constexpr int NC = GATED ? NR / 2 : NR, V = NR * MR;              // columns of the block, its sums
    constexpr int LEFT = V >= 16 ? V / 16 : 1, SHARE = V >= 16 ? 1 : 16 / V;      // sums a lane ends with; lanes with the same one
    __shared__ float red[WV * 4][V];
    __shared__ float squares[SCALED ? WV * 4 : 1][MR];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n0 = blockIdx.x * NC;
    // what the end needs beside the sums is asked for now: the result that this thread forms is (n, m); its share of the squares (of row t % MR)
    static_assert(!INTO || NC * MR <= 64, "one wave forms the results");
    const int t = threadIdx.x, n = t / MR, m = t % MR;
    const bool stores = t < NC * MR && m < M && n0 + n < N;
    const size_t at = (size_t)m * N + n0 + n;
    float before = 0.f, next = 0.f;
    if (INTO && stores) {
        before = C[at];
        next = fold.weight[n0 + n];
    }
    constexpr int SQ = 8, T = WV * 64;
    float sq[SCALED ? SQ : 1];
    if (SCALED) {
#pragma unroll
        for (int i = 0; i < SQ; ++i) sq[i] = t + T * i < fold.n_squares ? fold.squares_in[t + T * i] : 0.f;
    }
    const float* wrow[NR];
    const float* arow[MR];
#pragma unroll
    for (int n = 0; n < NR; ++n) wrow[n] = W + ((size_t)(n / NC) * N + min(n0 + n % NC, N - 1)) * K + 4 * lane;      // rows beyond N or M: the last row's, not stored
#pragma unroll
    for (int m = 0; m < MR; ++m) arow[m] = A + (size_t)min(m, M - 1) * K + 4 * lane;
    float acc[NR][MR] = {};
    struct Round { gf_f32x4_t w[U][NR], a[U][MR]; };
    auto fetch = [&](Round& f, int c) {                                // chunks c, c + WV, ...
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int n = 0; n < NR; ++n) f.w[u][n] = gf_stream(wrow[n] + (c + WV * u) * 256);
#pragma unroll
            for (int m = 0; m < MR; ++m) f.a[u][m] = gf_load(arow[m] + (c + WV * u) * 256);
        }
    };
    auto products = [&](const Round& f) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (int n = 0; n < NR; ++n)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[n][m] = fmaf(f.a[u][m][j], f.w[u][n][j], acc[n][m]);
    };
    auto single = [&](int k) {
        gf_f32x4_t w[NR];
#pragma unroll
        for (int n = 0; n < NR; ++n) w[n] = gf_stream(wrow[n] + k);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const gf_f32x4_t a = gf_load(arow[m] + k);
#pragma unroll
            for (int n = 0; n < NR; ++n)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[n][m] = fmaf(a[j], w[n][j], acc[n][m]);
        }
    };
    const int chunks = K >> 8, rounds = chunks / (WV * U);
    Round f0, f1;
    if (rounds > 0) {
        fetch(f0, wave);
        int i = 0;
        for (; i + 2 < rounds; i += 2) {
            fetch(f1, wave + (i + 1) * WV * U);
            products(f0);
            fetch(f0, wave + (i + 2) * WV * U);
            products(f1);
        }
        if (i + 1 < rounds) {
            fetch(f1, wave + (i + 1) * WV * U);
            products(f0);
            products(f1);
        } else {
            products(f0);
        }
    }
    int c = wave + rounds * WV * U;
    for (; c < chunks; c += WV) single(c * 256);
    if (c == chunks && chunks * 256 + 4 * lane < K) single(c * 256);      // the rest of K, a multiple of 4: the wave whose turn it is
    float sums[V];
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
        for (int m = 0; m < MR; ++m) sums[n * MR + m] = acc[n][m];
    gf_row_sums<V>(sums, lane);
    if (lane % SHARE == 0) {
#pragma unroll
        for (int i = 0; i < LEFT; ++i) red[wave * 4 + (lane >> 4)][(lane & 15) / SHARE * LEFT + i] = sums[i];
    }
    if (SCALED) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < SQ; ++i) s += sq[i];
        for (int i = t + T * SQ; i < fold.n_squares; i += T) s += fold.squares_in[i];
        s = gf_rotated_sum<0x128>(s);                          // lanes l and l + 8 of 16 (row_ror), ...
        if (MR <= 4) s = gf_rotated_sum<0x124>(s);
        if (MR <= 2) s = gf_rotated_sum<0x122>(s);
        if (MR <= 1) s = gf_rotated_sum<0x121>(s);
        if ((lane & 15) < MR) squares[wave * 4 + (lane >> 4)][lane & 15] = s;
    }
    __syncthreads();
    if (INTO ? wave > 0 : !stores) return;
    float y = 0.f, up = 0.f;
    if (!INTO || stores) {
#pragma unroll
        for (int p = 0; p < WV * 4; ++p) {
            y += red[p][t];
            if (GATED) up += red[p][t + V / 2];
        }
    }
    if (SCALED) {
        float s = 0.f;
#pragma unroll
        for (int p = 0; p < WV * 4; ++p) s += squares[p][m];
        const float scale = 1.0f / sqrtf(s / (float)K + fold.eps);
        y *= scale;
        up *= scale;
    }
    if (GATED) y = gated_value(act, y, up);
    if (!INTO) {
        C[at] = y;
        return;
    }
    y += before;                                               // (lanes that store nothing: zero)
    if (stores) {
        C[at] = y;
        fold.rows_out[at] = y * next;
    }
    float s = y * y;
#pragma unroll
    for (int o = MR; o < NC * MR; o <<= 1) s += __shfl_xor(s, o, 64);
    if (t < MR) fold.squares_out[(size_t)blockIdx.x * MR + t] = s;
}

// ---- a few tiles of rows ----------------------------------------------------------------------------------------------------
#define GF_WAVES 8
template <int MT>
__global__ __launch_bounds__(GF_WAVES * 64) void gemm_f32_narrow_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                        float* __restrict__ C, int M, int N, int K) {
    __shared__ float red[GF_WAVES][MT][64][4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    A += (size_t)blockIdx.y * (16 * MT) * K;
    C += (size_t)blockIdx.y * (16 * MT) * N;
    M -= blockIdx.y * (16 * MT);
    const float* wrow = W + (size_t)min(n0 + r, N - 1) * K + 4 * g;
    const float* arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) arow[mt] = A + (size_t)min(mt * 16 + r, M - 1) * K + 4 * g;
    gf_f32x4_t acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](gf_f32x4_t (&w)[4], gf_f32x4_t (&a)[MT][4], int k) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            w[s] = gf_stream(wrow + k + 16 * s);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) a[mt][s] = gf_load(arow[mt] + k + 16 * s);
        }
    };
    auto products = [&](const gf_f32x4_t (&w)[4], const gf_f32x4_t (&a)[MT][4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s][j], a[mt][s][j], acc[mt], 0, 0, 0);
    };
    // two sets of operands taken in turn: the next chunk's are asked for before this chunk's products
    const int chunks = K >> 6, mine = (chunks - wave + GF_WAVES - 1) / GF_WAVES;
    gf_f32x4_t w0[4], a0[MT][4], w1[4], a1[MT][4];
    if (mine > 0) {
        auto at = [&](int i) { return (wave + i * GF_WAVES) * 64; };
        fetch(w0, a0, at(0));
        int i = 0;
        for (; i + 2 < mine; i += 2) {
            fetch(w1, a1, at(i + 1));
            products(w0, a0);
            fetch(w0, a0, at(i + 2));
            products(w1, a1);
        }
        if (i + 1 < mine) {
            fetch(w1, a1, at(i + 1));
            products(w0, a0);
            products(w1, a1);
        } else {
            products(w0, a0);
        }
    }
    if (wave == (chunks & (GF_WAVES - 1))) {              // the rest of K: the wave whose turn it would be
        for (int k = chunks * 64; k < K; k += 16) {
            const bool ok = k + 4 * g < K;
            const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
            const gf_f32x4_t w = ok ? gf_stream(wrow + k) : zero;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const gf_f32x4_t a = ok ? gf_load(arow[mt] + k) : zero;
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], a[j], acc[mt], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<gf_f32x4_t*>(red[wave][mt][lane]) = acc[mt];
    __syncthreads();
    if (wave >= MT) return;
    // row tile mt is summed, in the order of the waves, and stored by wave mt: lane (r, g) has C[row r][columns 4 g ..]
    gf_f32x4_t sum = *reinterpret_cast<const gf_f32x4_t*>(red[0][wave][lane]);
#pragma unroll
    for (int w = 1; w < GF_WAVES; ++w) sum += *reinterpret_cast<const gf_f32x4_t*>(red[w][wave][lane]);
    const int m = wave * 16 + r;
    if (m >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n0 + 4 * g + i < N) C[(size_t)m * N + n0 + 4 * g + i] = sum[i];
}

// ---- up to 32 rows, plenty of rows of W ------------------------------------------------------------------------------------------
// Bound by W from memory, as few rows are, but with the matrix cores' arithmetic, and without the narrow kernel's reading of A once per 16
// rows of W (as many bytes as W from 16 rows on: there 16 rows cost more than 9 at the same products).  A block of eight waves stays on its
// compute unit: each wave keeps its eighth of K of all of A in registers (16 CH a row tile; CH chunks of 64 of K) and goes through every
// so many-th tile of 16 rows of W, a chunk's registers filled for the next tile as soon as its products are done.  Waves add through LDS,
// one barrier a tile.  `parts` parts of K go to blocks of their own, for results too narrow to give every compute unit a tile: C
// [parts][M][N].  GATED: a tile is 8 rows of the gate and the same 8 of the other half.  us, the kernels it stands for / this, at 16 and at 32 rows:
// 12288 x 2048 43 / 24.5 and 43 / 31, with its activation 45 / 23.5 and 45 / 29; 32768 x 2048 84 / 55 and 84 / 66; 151936 x 1024 196 / 144 and 196 /
// 157 (8 rows 187 / 132); 6144 x 1024 11.6 / 9.9 and 15.2 / 13.6; in parts of 512 of K 1024 x 2048 10.1 / 4.9 and 7.7 / 6.0, 2048 x 6144 27.8 /
// 14.1 and 21.9 / 18.9, 2560 x 4096 18.6 / 11.5 and 18.7 / 15.3.
#define GF_HELD_WAVES 8
template <int MT, int CH, bool GATED>
__global__ __launch_bounds__(GF_HELD_WAVES * 64) void gemm_f32_held_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                           float* __restrict__ C, int M, int N, int K, int parts, GateAct act) {
    constexpr int NC = GATED ? 8 : 16;                                            // columns of a tile
    __shared__ float red[2][GF_HELD_WAVES][MT][64][4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int part = blockIdx.x % parts, step = gridDim.x / parts, tiles = (N + NC - 1) / NC;
    const int k0 = (part * GF_HELD_WAVES + wave) * 64 * CH + 4 * g;
    C += (size_t)part * M * N;
    int t = blockIdx.x / parts, turn = 0;
    gf_f32x4_t w[CH][4], a[MT][CH][4], acc[MT];
    auto row_of = [&](int t) {                                                    // rows beyond N or M: the last row's, not stored
        const int n = min(t * NC + r % NC, N - 1);
        return W + (size_t)(GATED && r >= NC ? N + n : n) * K + k0;
    };
    const float* wrow = row_of(t);
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int s = 0; s < 4; ++s) w[c][s] = gf_stream(wrow + c * 64 + 16 * s);
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int s = 0; s < 4; ++s) a[mt][c][s] = gf_load(A + (size_t)min(mt * 16 + r, M - 1) * K + k0 + c * 64 + 16 * s);
    auto tile = [&](auto more) {
        if (more) wrow = row_of(t + step);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < CH; ++c) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[c][s][j], a[mt][c][s][j], acc[mt], 0, 0, 0);
            if (more) {                                                           // the next tile's, as soon as this chunk's registers are free
#pragma unroll
                for (int s = 0; s < 4; ++s) w[c][s] = gf_stream(wrow + c * 64 + 16 * s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the waves' sums meet in one of two places; a wave that writes one again has passed the barrier behind its last reader
        float (&to)[GF_HELD_WAVES][MT][64][4] = red[turn & 1];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<gf_f32x4_t*>(to[wave][mt][lane]) = acc[mt];
        __syncthreads();
        const int mt = (wave - turn * MT) & (GF_HELD_WAVES - 1);                   // (the waves take turns to add)
        if (mt < MT) {
            // lane (r, g) has C[row r][columns 4 g ..]; gated: columns 4 g .. of the gate for g < 2, lane + 32 the same of the other
            gf_f32x4_t sum = *reinterpret_cast<const gf_f32x4_t*>(to[0][mt][lane]);
#pragma unroll
            for (int v = 1; v < GF_HELD_WAVES; ++v) sum += *reinterpret_cast<const gf_f32x4_t*>(to[v][mt][lane]);
            if constexpr (GATED) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float up = __shfl_xor(sum[i], 32, 64);
                    sum[i] = gated_value(act, sum[i], up);
                }
            }
            const int m = mt * 16 + r;
            if (m < M && 4 * g < NC) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t * NC + 4 * g + i < N) C[(size_t)m * N + t * NC + 4 * g + i] = sum[i];
            }
        }
    };
    for (; t + step < tiles; t += step, ++turn) tile(std::true_type{});
    tile(std::false_type{});
}

// ---- many rows ----------------------------------------------------------------------------------------------------------------
// A tile of 64 x 64 of C per 256 threads, a wave a quarter of it (v_mfma_f32_32x32x2_f32, 64 cycles each).  Steps of 32 of K: two
// steps' pieces of A and W are on their way to registers while this one's products run from LDS, two LDS stages, one barrier a
// step.  Rows are padded to 36 floats: eight neighbouring rows start in different groups of four banks.  A wave's operands are 2 KB
// of LDS per 256 cycles of products, a quarter of what LDS gives.  KS > 1: so many groups of 256 threads share a tile, each a part
// of K.  Tiles of 128 x 128 were no faster (611 rows, 12288 x 2048: 308 against 304 us) and leave small products fewer blocks.
// Measured: 102 TFLOP/s at 611 rows of 12288 x 2048, 110 at 1200 (the library's own float32 product gets 134 at 4096^3, the chip's
// nominal rate is 157); the plain FMA kernel it stands for 10.
#define GF_BK 32
#define GF_LD 36
template <int KS>
__global__ __launch_bounds__(256 * KS) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                                                                 int M, int N, int K, int tiles_m, int tiles_n, int parts) {
    __shared__ float lds[KS][2][128 * GF_LD];         // per part of K two stages: 64 rows of A, then 64 of W
    // blocks go to the eight dies in turn: die x takes a run of neighbouring tiles, rows fastest, so that a piece of W is read into one L2
    const int tiles = tiles_m * tiles_n, total = tiles * parts, per = (total + 7) >> 3;
    const int at = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || at >= total) return;
    const int tile = at % tiles, k_part = at / tiles;
    C += (size_t)k_part * M * N;
    const int m0 = (tile % tiles_m) * 64, n0 = (tile / tiles_m) * 64;
    const int part = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, tid = threadIdx.x & 255;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = threadIdx.x & 63;
    const int i = lane & 31, h = lane >> 5;
    const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
    // staging: thread t has rows t / 8 and t / 8 + 32, values 4 (t % 8) .. of the step: eight lanes read 128 bytes of one row
    const int sr = tid >> 3, sk = (tid & 7) * 4;
    const float* ap[2];
    const float* wp[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        ap[p] = A + (size_t)min(m0 + sr + 32 * p, M - 1) * K;       // rows beyond M or N: the last row's, not stored
        wp[p] = W + (size_t)min(n0 + sr + 32 * p, N - 1) * K;
    }
    // this part's steps of K: `steps` for every part (the barriers are the block's), those from its end on staged as zeros
    const int all_steps = (K + GF_BK - 1) / GF_BK, step0 = (int)((long long)all_steps * k_part / parts);
    const int all = (int)((long long)all_steps * (k_part + 1) / parts) - step0, steps = (all + KS - 1) / KS;
    const int k_last = min(K, (step0 + all) * GF_BK);
    const int k_first = (step0 + part * steps) * GF_BK, k_end = min(k_last, k_first + steps * GF_BK);
    const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    auto fetch = [&](gf_f32x4_t (&va)[2], gf_f32x4_t (&vw)[2], int s) {
        const int k = min(k_first + s * GF_BK + sk, K - 4);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            va[p] = gf_load(ap[p] + k);
            vw[p] = gf_load(wp[p] + k);
        }
    };
    auto stage = [&](const gf_f32x4_t (&va)[2], const gf_f32x4_t (&vw)[2], int s) {
        const bool in = k_first + s * GF_BK + sk < k_end;
        float* to = lds[part][s & 1] + sr * GF_LD + sk;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            *reinterpret_cast<gf_f32x4_t*>(to + 32 * p * GF_LD) = in ? va[p] : zero;
            *reinterpret_cast<gf_f32x4_t*>(to + (64 + 32 * p) * GF_LD) = in ? vw[p] : zero;
        }
    };
    // A sum over all of K in one chain would round K times: every 256 of K the chain's value goes to a second sum (611 x 1024 x 3072:
    // relative error 2.9e-7 against 1.0e-6 for one chain)
    gf_f32x16_t acc, sum;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = sum[e] = 0.f;
    auto products = [&](int s) {
        const float* fa_at = lds[part][s & 1] + (wm + i) * GF_LD + 4 * h;
        const float* fw_at = lds[part][s & 1] + (64 + wn + i) * GF_LD + 4 * h;
#pragma unroll
        for (int kk = 0; kk < GF_BK; kk += 8) {
            const gf_f32x4_t fa = gf_load(fa_at + kk), fw = gf_load(fw_at + kk);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[j], fa[j], acc, 0, 0, 0);
        }
        if ((s & 7) == 7 || s + 1 == steps) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                sum[e] += acc[e];
                acc[e] = 0.f;
            }
        }
    };
    // step s runs from LDS stage s & 1 while the pieces of steps s + 1 and s + 2 are on their way (steps beyond the last read the
    // last values of K again); a stage written behind step s was read last in step s - 1, which every wave left at a barrier
    gf_f32x4_t a0[2], v0[2], a1[2], v1[2];
    fetch(a0, v0, 0);
    fetch(a1, v1, 1);
    stage(a0, v0, 0);
    __syncthreads();
    int s = 0;
    for (; s + 2 < steps; s += 2) {
        fetch(a0, v0, s + 2);
        products(s);
        stage(a1, v1, s + 1);
        __syncthreads();
        fetch(a1, v1, s + 3);
        products(s + 1);
        stage(a0, v0, s + 2);
        __syncthreads();
    }
    products(s);
    if (s + 1 < steps) {
        stage(a1, v1, s + 1);
        __syncthreads();
        products(s + 1);
    }
    if (KS > 1) {
        // the other parts' sums through LDS (their own stages) to the first part's waves, added in the order of the parts
        __syncthreads();
        float* mine = lds[part][0] + wave * 1024 + 4 * lane;
        if (part > 0) {
#pragma unroll
            for (int e = 0; e < 16; e += 4) *reinterpret_cast<float4*>(mine + e * 64) = make_float4(sum[e], sum[e + 1], sum[e + 2], sum[e + 3]);
        }
        __syncthreads();
        if (part > 0) return;
#pragma unroll
        for (int p = 1; p < KS; ++p)
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
                const float4 v = *reinterpret_cast<const float4*>(lds[p][0] + wave * 1024 + 4 * lane + e * 64);
                sum[e] += v.x; sum[e + 1] += v.y; sum[e + 2] += v.z; sum[e + 3] += v.w;
            }
    }
    // lane (i, h) has C[row i][columns 8 q + 4 h .. + 3], q < 4
    const int m = m0 + wm + i;
    if (m >= M) return;
    const bool whole = (N & 3) == 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn + 8 * q + 4 * h;
        float* to = C + (size_t)m * N + n;
        if (whole) {
            if (n < N) *reinterpret_cast<float4*>(to) = make_float4(sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < N) to[e] = sum[4 * q + e];
        }
    }
}

// ---- dispatch --------------------------------------------------------------------------------------------------------------
bool gemm_f32_takes(const void* A, const void* W, const void* C, int M, int N, int K) {
    const uintptr_t at = (uintptr_t)A | (uintptr_t)W | (uintptr_t)C;
    return K % 4 == 0 && at % 16 == 0 && (int64_t)((N + 63) / 64) * ((M + 63) / 64) < (1 << 28);
}

// Up to 8 rows; from 5 on not 4096 rows of W and more with a K up to 1024, whose blocks have little to stream (8 rows, 4096 x 1024: 7.3 us,
// the narrow kernel 6.9; 4096 x 2048 10.1 / 11.0).
static bool gf_few_takes(int M, int N, int K) { return M <= 4 || (M <= 8 && (N < 4096 || K > 1024)); }

// Rows of W a block, and waves: eight rows where there are plenty (4 rows of A: 12288 x 2048 gated 18.3 us, with four 19.5; 2048 x 6144 11.5 / 10.6;
// 8 rows of A: 4096 x 2048 10.1 / 10.9), and up to 1024 rows of W eight waves a block to have enough of them (4 rows of A, 1024 x 3072 5.0
// us, four waves 5.7) or, for two rows of A, two rows of W (1024 x 2048 3.7 / 3.6, 1024 x 3072 4.6 / 4.4).  One row of A costs little to bring
// again, and up to 4 million numbers of W blocks of one row are the fastest, a chunk a wave and round (what stood before / two rows, or four beyond
// 1024 of W / one): 1024 x 1024 2.76 / 2.79 / 2.74, 1024 x 2048 3.50 / 3.44 / 3.38, 1024 x 3072 4.05 / 4.23 / 3.94, 1024 x 4096 5.15 / 4.81 / 4.64, 2048 x 2048
// 4.65 / 4.72 / 4.57, 4096 x 1024 4.93 / 4.75 / 4.70; beyond, 2048 x 3072 four 5.78, one 6.16, 4096 x 2048 7.35 / 7.12 / 7.40.  Below 1024 rows of W two
// chunks a round, where that leaves no rest: 512 x 2048 2.68, one 2.96 (two rows of W 2.78); 256 x 2048 2.34, 2.69 (2.50); 512 x 3072 3.26, 3.14 (3.40).
// With `blocks` given nothing runs, and it becomes the number of blocks.
template <bool GATED, bool SCALED = false, bool INTO = false>
static void gf_few(const float* A, const float* W, float* C, int M, int N, int w_rows, int K, GateAct act, hipStream_t st, const GfFold& fold = GfFold{}, int* blocks = nullptr) {
#define GF_FEW(MR, NR, U, WV)                                                                                                      \
    {                                                                                                                              \
        const int grid = (N + NR / (GATED ? 2 : 1) - 1) / (NR / (GATED ? 2 : 1));                                                  \
        if (blocks) *blocks = grid;                                                                                                \
        else gemm_f32_few_kernel<MR, NR, U, WV, GATED, SCALED, INTO><<<grid, WV * 64, 0, st>>>(A, W, C, M, N, K, act, fold);       \
    }
    if constexpr (!GATED) {
        if (M == 1 && (int64_t)w_rows * K <= (4 << 20)) {
            if (w_rows < 1024 && K % 2048 == 0) GF_FEW(1, 1, 2, 4) else GF_FEW(1, 1, 1, 4)
            return;
        }
    }
    if (M == 1) { if (w_rows <= 1024) GF_FEW(1, 2, 2, 4) else GF_FEW(1, 4, 2, 4) }
    else if (M == 2) { if (w_rows <= 1024) GF_FEW(2, 2, 2, 4) else GF_FEW(2, 4, 2, 4) }
    else if (M <= 4) { if (w_rows <= 1024) GF_FEW(4, 4, 1, 8) else if (w_rows < 8192) GF_FEW(4, 4, 1, 4) else GF_FEW(4, 8, 1, 4) }
    else { if (w_rows <= 1024) GF_FEW(8, 4, 1, 8) else if (w_rows < 4096) GF_FEW(8, 4, 1, 4) else GF_FEW(8, 8, 1, 4) }
#undef GF_FEW
}

// K (or a part of it) ends at 2048 because a wave's registers do: a chunk of 64 takes 16 of them for W and 16 for each row tile, and with two row
// tiles four chunks leave room in 256, five do not.  (One row tile would fit K = 3072; it is not built: in parts o and down of a wider model are
// taken, its gate/up and head stay with the narrow kernel.)
static bool gf_held_takes(int M, int N, int K, int parts) { return M <= 32 && N < (1 << 30) && K % (512 * parts) == 0 && K / parts <= 2048; }

// a block for each compute unit: another one brings A's values again and takes no part of the memory's time (12288 x 2048, 16 rows 24.5 us, two
// blocks 28.9; 32 rows 31 / 40)
template <bool GATED>
static void gf_held(const float* A, const float* W, float* C, int M, int N, int K, int parts, GateAct act, hipStream_t st) {
    const int tiles = (N + (GATED ? 7 : 15)) / (GATED ? 8 : 16), grid = parts * min(tiles, max(1, 256 / parts)), ch = K / parts / 512;
#define GF_HELD(MT, CH) gemm_f32_held_kernel<MT, CH, GATED><<<grid, GF_HELD_WAVES * 64, 0, st>>>(A, W, C, M, N, K, parts, act)
    if (M <= 16) { if (ch == 1) GF_HELD(1, 1); else if (ch == 2) GF_HELD(1, 2); else if (ch == 3) GF_HELD(1, 3); else GF_HELD(1, 4); }
    else { if (ch == 1) GF_HELD(2, 1); else if (ch == 2) GF_HELD(2, 2); else if (ch == 3) GF_HELD(2, 3); else GF_HELD(2, 4); }
#undef GF_HELD
}

int gemm_f32(const float* A, const float* W, float* C, int M, int N, int K, hipStream_t st) {
#define GF_NARROW(MT) gemm_f32_narrow_kernel<MT><<<dim3(tiles16, (M + 16 * MT - 1) / (16 * MT)), GF_WAVES * 64, 0, st>>>(A, W, C, M, N, K)
#define GF_TILE(KS) gemm_f32_tile_kernel<KS><<<((tm * tn + 7) / 8) * 8, 256 * KS, 0, st>>>(A, W, C, M, N, K, tm, tn, 1)
    const int tiles16 = (N + 15) / 16, tm = (M + 63) / 64, tn = (N + 63) / 64;
    if (gemm_f32_split_takes(M, N, K, 1)) return gemm_f32_split(A, W, C, M, N, K, 1, st);
    if (gf_few_takes(M, N, K)) {
        gf_few<false>(A, W, C, M, N, N, K, GateAct{1.f, 0.f}, st);
    } else if (gf_held_takes(M, N, K, 1) && N > 4096) {
        // (from the first size on that gives a compute unit two tiles: 4112 x 1024, 16 rows, the narrow kernel 10.7 us, this 9.3, 32 rows 14.1 / 12.2,
        // 4112 x 2048 17.9 / 16.0 and 25.0 / 21.4; with one tile a unit 4096 x 1024 7.4 / 7.6 and 9.1 / 11.0)
        gf_held<false>(A, W, C, M, N, K, 1, GateAct{1.f, 0.f}, st);
    } else if (tm * tn < 160) {
        // Row tiles per block: as many as leave a block for every compute unit, W being read once per group of them (24 rows, 2048 x
        // 2048: 10.4 us with one, 13.1 with two; 4096 x 2048: 19.4 with one, 14.5 with two; 64 rows, 4096 x 1024: 20 / 15.3 / 13.9
        // with one / two / four).  Up to 64-row tiles for 160 blocks this kernel is ahead of the next (64 rows, 6144 x 1024: 22.6
        // against 24.6 us; 200 rows, 1024 x 2048: 21.5 / 40.7; behind it at 64 rows, 12288 x 2048: 68 / 49 and at 300, 2048 x 2048: 58 / 42).
        if (M > 32 && tiles16 * ((M + 63) / 64) >= 256) GF_NARROW(4);
        else if (M > 16 && tiles16 * ((M + 31) / 32) >= 256) GF_NARROW(2);
        else GF_NARROW(1);
    } else {
        // Parts of K in a block: where a compute unit has one or two blocks, more waves hide the loads, LDS and barriers of each
        // other (611 rows, 1024 x 2048, 160 blocks: 51.6 / 43.8 / 41.1 us with one / two / four; 300 rows, 4096 x 2048, 320 blocks:
        // 80.9 / 76.8 / 80.2; 1200 rows, 12288 x 2048: 550 / 556 / 596).
        if (tm * tn <= 256) GF_TILE(4);
        else if (tm * tn <= 512) GF_TILE(2);
        else GF_TILE(1);
    }
    SPY_CHECK_LAUNCH("spy_gemm (float32)");
    return 0;
}

// act(A . Wgate^T) * (A . Wup^T) for up to eight rows, up to 32 where A is held, and for those that gemm_f32_split.hip takes, W = [gate rows | up rows] of N each, without the [M][2 N] result in between.
extern "C" int spy_gemm_f32_gated(float* C, const float* A, const float* W, int M, int N, int K, int act_code, hipStream_t st) {
    GateAct act;
    SPY_REQUIRE(M > 0 && N > 0 && K > 0 && gate_act_of(act_code, &act), "spy_gemm_f32_gated: %d rows, activation %d", M, act_code);
    SPY_REQUIRE(gemm_f32_takes(A, W, C, M, N, K), "spy_gemm_f32_gated: operands of %d x %d x %d are not taken", M, N, K);
    const bool held = M > 8 && gf_held_takes(M, N, K, 1);
    SPY_REQUIRE(M <= 8 || held || (N < (1 << 30) && gemm_f32_split_takes(M, 2 * N, K, 1)), "spy_gemm_f32_gated: %d rows of %d x %d are not taken", M, N, K);
    if (held) gf_held<true>(A, W, C, M, N, K, 1, act, st);
    else if (M > 8) return gemm_f32_split_gated(A, W, C, M, 2 * N, K, act, st);
    else gf_few<true>(A, W, C, M, N, 2 * N, K, act, st);
    SPY_CHECK_LAUNCH("spy_gemm_f32_gated");
    return 0;
}

// A [M, K] . W [N, K]^T in parts of K: C [parts][M][N], a block a tile of one part, which the reader sums (spy_add_parts_rmsnorm).  For
// results whose tiles fill no whole number of rounds of the chip (or of which there are too few even for that: the narrow kernel above
// reads half lines of W).  Parts beat groups of a block's waves, which leave the other compute units idle.  Measured, us, the
// kernels above / this one and what the sum adds to the norm's pass: 17 rows, 2560 x 4096 29 / 18.5 + 1; with gemm_f32_split.hip's blocks: 611
// rows, 1024 x 2048 43 / 21.4 + 2, 1024 x 3072 63 / 28 + 5; 90 rows, 2048 x 2048 22 / 12.6 + 1.
extern "C" int spy_gemm_f32_parts(float* C, const float* A, const float* W, int M, int N, int K, int parts, hipStream_t st) {
    SPY_REQUIRE(M > 0 && N > 0 && K > 0 && parts >= 1 && parts <= (K + GF_BK - 1) / GF_BK, "spy_gemm_f32_parts: %d parts of %d x %d x %d", parts, M, N, K);
    SPY_REQUIRE(gemm_f32_takes(A, W, C, M, N, K), "spy_gemm_f32_parts: operands of %d x %d x %d are not taken", M, N, K);
    if (parts <= K / GF_BK && gemm_f32_split_takes(M, N, K, parts)) return gemm_f32_split(A, W, C, M, N, K, parts, st);
    if (gf_held_takes(M, N, K, parts)) {
        gf_held<false>(A, W, C, M, N, K, parts, GateAct{1.f, 0.f}, st);
        SPY_CHECK_LAUNCH("spy_gemm_f32_parts");
        return 0;
    }
    const int tm = (M + 63) / 64, tn = (N + 63) / 64;
    const int64_t blocks = (int64_t)tm * tn * parts;
    SPY_REQUIRE(blocks < (1 << 28), "spy_gemm_f32_parts: too many blocks");
    gemm_f32_tile_kernel<1><<<(unsigned)((blocks + 7) / 8 * 8), 256, 0, st>>>(A, W, C, M, N, K, tm, tn, parts);
    SPY_CHECK_LAUNCH("spy_gemm_f32_parts");
    return 0;
}

// Parts of a row's squares that the product into the stream writes: one a block, [parts][rows rounded up to a power of two]
extern "C" int spy_gemm_f32_into_parts(int M, int N, int K) {
    int blocks = 0;
    if (M > 0 && M <= 8 && N > 0 && K > 0) gf_few<false, false, true>(nullptr, nullptr, nullptr, M, N, N, K, GateAct{1.f, 0.f}, nullptr, GfFold{}, &blocks);
    return blocks;
}

// C (the stream, [M, N]) += A . W^T for up to eight rows; rows_out = C weight; squares: see gemm_f32_few_kernel, `parts` of them.
extern "C" int spy_gemm_f32_into(float* C, const float* A, const float* W, float* rows_out, const float* weight, float* squares, int parts, int M, int N, int K,
                                 hipStream_t st) {
    SPY_REQUIRE(M > 0 && M <= 8 && N > 0 && K > 0 && parts == spy_gemm_f32_into_parts(M, N, K), "spy_gemm_f32_into: %d rows, %d parts", M, parts);
    SPY_REQUIRE(gemm_f32_takes(A, W, C, M, N, K), "spy_gemm_f32_into: operands of %d x %d x %d are not taken", M, N, K);
    gf_few<false, false, true>(A, W, C, M, N, N, K, GateAct{1.f, 0.f}, st, GfFold{nullptr, 0, 0.f, rows_out, weight, squares});
    SPY_CHECK_LAUNCH("spy_gemm_f32_into");
    return 0;
}

// The products of such rows [M, K], up to eight: C [M, N] = A . W^T scaled by row, or, gated, act(gate) * up of that, W = [gate rows | up rows] of N each.
extern "C" int spy_gemm_f32_scaled(float* C, const float* A, const float* W, const float* squares, int parts, float eps, int M, int N, int K, int gated, int act_code,
                                   hipStream_t st) {
    GateAct act = {1.f, 0.f};
    SPY_REQUIRE(M > 0 && M <= 8 && N > 0 && K > 0 && parts > 0 && parts <= (1 << 24), "spy_gemm_f32_scaled: %d rows, %d parts", M, parts);
    SPY_REQUIRE(!gated || gate_act_of(act_code, &act), "spy_gemm_f32_scaled: activation %d", act_code);
    SPY_REQUIRE(gemm_f32_takes(A, W, C, M, N, K), "spy_gemm_f32_scaled: operands of %d x %d x %d are not taken", M, N, K);
    const int MR = M <= 2 ? M : M <= 4 ? 4 : 8;
    const GfFold fold = {squares, parts * MR, eps, nullptr, nullptr, nullptr};
    if (gated) gf_few<true, true>(A, W, C, M, N, 2 * N, K, act, st, fold);
    else gf_few<false, true>(A, W, C, M, N, N, K, act, st, fold);
    SPY_CHECK_LAUNCH("spy_gemm_f32_scaled");
    return 0;
}
