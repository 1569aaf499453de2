// Products of many float32 rows, C[M, N] = A[M, K] . W[N, K]^T, on the matrix cores' bfloat16 instructions, which multiply sixteen times
// as much in a cycle as their float32 ones do.  Every value is cut into three bfloat16 parts, x = high + middle + low (8 + 8 + 8
// bits, each part the rounded rest of those before it), a product of two parts is exact in float32, and of the nine products of parts
// the six from 2^-18 of the result on are formed: high high apart, high middle, middle high, middle middle, high low and low high
// in a second sum.  What is left out is at most 2^-24 of |a||w|, one rounding in float32 (middle parts are up to 2^-8 of a value, low ones
// 2^-17), and 2^-27.4 in the root of the mean square.  Relative errors against 64 bits (2-norm, normal
// values): K = 1024 1.9e-7, K = 2048 2.7e-7, in parts less; the float32 instructions' 2.9e-7 (gemm_f32.hip, whose chain ends every 256 of K).
// The cut loses nothing down to about 2^-110, where low parts meet bfloat16's smallest number; sums with smaller values, infinities, NaN or what
// bfloat16 rounds to infinity are formed by float32 instructions (at the end).
// GATED: W = [gate rows | up rows], C[M][N / 2] = act(gate) * up.
//
// Three of the six are of W's middle and low parts, which are zero where a matrix is a bfloat16 checkpoint's, widened: a block begins
// without them, keeps the low halves' bits of all that it stages of W, and looks at them behind its first step, every eighth and its last.  If
// any is set, what the steps since the last look left out is added and the others are formed with all six.  Rows of W without such bits have the
// same sums bit for bit either way; nothing about a matrix is kept from one block or call to the next.  Measured, us, a widened matrix / one of
// float32 values / widened but for its last 32 of K / for its second half: 611 rows, 4096 x 1024 30.0 / 41 / 38 / 44, 6144 x 1024 gated 34 / 50 / 42.5 /
// 51; 400 rows, 4096 x 2048 43.5 / 61 / 48.5 / 56, 12288 x 2048 gated 106 / 162 / 125 / 149; 90 rows, 4096 x 2048 30.5 / 38.4 / 34.8 / 39.1 (tiles anew from the
// start cost 61.6, 72, 91, 240 and 64 for the last two).  A look behind each step, and on from there, took 2 to 3 us of a widened 4096 x 1024.
//
// A block splits its rows of A and W as it stages them: from memory into registers four steps of 32 of K ahead, from there as three planes
// in operand order into the other of two LDS stages, while this step's products run.  128 x 128 values of C and eight waves
// (two a SIMD, one block a compute unit) where the tiles fill the chip, else 64 x 64 and four waves, two blocks a compute unit.
// What bounds it: a step of the large tile is 1536 cycles of products a SIMD and about 700 of the split (5.5 instructions a value), of which
// the matrix cores' work hides less than half; it takes 1.0 us.  The split by v_dot2_f32_bf16 (3.5 instructions a value) was slower beside
// MFMAs, and loads two steps ahead cost a third of the time (1.25 us).
// Measured, us, gemm_f32.hip's float32 instructions / this: 611 rows, 4096 x 1024 67 / 44, 6144 x 1024 87 / 49 (157 TFLOP/s), 1024 x 3072 in
// parts 44 / 28; 200 rows, 12288 x 2048 124 / 78, 2048 x 6144 in parts 61 / 38; 90 rows, 12288 x 2048 81 / 57.
#include "gemm_f32.h"
#include <type_traits>

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gs_f32x4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float gs_f32x16_t;
typedef __bf16 gs_bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 gs_bf16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t gs_u32x4_t;

#define GS_BK 32
#define GS_PIECE 576          // bytes of 32 rows of 8 values of K in one plane, 64 of them unused
#define GS_GROUP (4 * GS_PIECE)

// Middle and low parts of what is left of two values behind their high ones.  What the low part is rounded from has eight bits at most and the
// same smallest exponent as a bfloat16, so nothing is lost unless its 24 - 8 last bits are beyond that exponent: those bits go to `lost`.
__device__ __forceinline__ void gs_split_rest(float x0, float x1, uint32_t& m, uint32_t& l, uint32_t& lost) {
    m = pack_bf16x2(x0, x1);
    x0 -= __uint_as_float(m << 16);
    x1 -= __uint_as_float(m & 0xffff0000u);
    l = pack_bf16x2(x0, x1);
    lost |= __float_as_uint(x0) | __float_as_uint(x1);
}
// x = high + middle + low, each a bfloat16, two values at a time
__device__ __forceinline__ void gs_split(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l, uint32_t& lost) {
    h = pack_bf16x2(x0, x1);
    gs_split_rest(x0 - __uint_as_float(h << 16), x1 - __uint_as_float(h & 0xffff0000u), m, l, lost);
}

template <int BM, int BN, int WM, int WN, bool GATED>
__global__ __launch_bounds__(64 * WM * WN) void gemm_f32_split_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                                                                      int M, int N, int K, int tiles_m, int tiles_n, int parts, GateAct act) {
    constexpr int T = 64 * WM * WN, MT = BM / WM / 32, NT = BN / WN / 32, ROWS = T / 4, P = (BM + BN) / ROWS;
    constexpr int PLANE = (BM + BN) / 32 * GS_GROUP, STAGE = 3 * PLANE;
    static_assert(BM % ROWS == 0 && BN % ROWS == 0, "a thread's piece is of A or of W for the whole block");
    __shared__ __align__(16) char lds[2 * STAGE];
    __shared__ uint32_t no_bf16;                       // whether a value of W is no bfloat16 number
    const int tiles = tiles_m * tiles_n, total = tiles * parts, per = (total + 7) >> 3;
    const int at = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || at >= total) return;
    const int tile = at % tiles, k_part = at / tiles;
    C += (size_t)k_part * M * N;                       // (parts are of the product alone, not of a gated one)
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int i = lane & 31, h = lane >> 5;
    const int wm = wave % WM, wn = wave / WM;
    // W's row in place `at` of the block's BN (one that does not exist reads the last; nothing is stored).  GATED: of 32 places 16 are gate
    // rows and 16 the up rows of the same columns, so that a lane has both values of a column
    auto w_row = [&](int at) {
        if (!GATED) return min(n0 + at, N - 1);
        return min(n0 / 2 + (at >> 5) * 16 + (at & 15), N / 2 - 1) + ((at & 16) ? N / 2 : 0);
    };
    // staging: thread t has eight values of rows t / 4, t / 4 + ROWS, ...; four threads read 128 bytes of one row
    const int sr = tid >> 2, kp = tid & 3;
    const auto ares = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, M * K * 4, 0x00020000);
    const auto wres = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, N * K * 4, 0x00020000);
    int src[P], dst[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int row = sr + p * ROWS;
        src[p] = ((p * ROWS < BM ? min(m0 + row, M - 1) : w_row(row - BM)) * K + kp * 8) * 4;
        dst[p] = (row >> 5) * GS_GROUP + kp * GS_PIECE + (row & 31) * 16;
    }
    const int all_steps = K / GS_BK, part0 = (int)((long long)all_steps * k_part / parts), part1 = (int)((long long)all_steps * (k_part + 1) / parts);
    int step0 = part0, steps = part1 - part0;          // what is still to do of the part
    struct Pieces { gs_f32x4_t v[P][2]; };
    auto fetch = [&](Pieces& f, int s) __attribute__((always_inline)) {
        const int k = (step0 + min(s, steps - 1)) * GS_BK * 4;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                f.v[p][e] = __builtin_bit_cast(gs_f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(p * ROWS < BM ? ares : wres, src[p] + 16 * e, k, 0));
        __builtin_amdgcn_sched_barrier(0);
    };
    // Ways to form a step.  WHOLE: W's values are taken to be bfloat16 numbers, whose middle and low parts are zero; `rest` keeps the bits that
    // say otherwise.  FULL: all six products.  REST: what WHOLE left out of a step where it does say otherwise: its high part is the value cut off
    // behind 16 bits, so that the middle part here is up to 2^-7 of the value, and its product with A's low part comes along.
    enum Way { WHOLE, FULL, REST };
    uint32_t rest = 0, lost[P] = {};
    auto stage = [&](Pieces& f, int s, auto way) __attribute__((always_inline)) {
        constexpr int WAY = decltype(way)::value;
        char* to = lds + (s & 1) * STAGE;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            gs_u32x4_t hi, mid, lo;
            const bool cut = WAY != FULL && p * ROWS >= BM;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x0 = f.v[p][e >> 1][(e & 1) * 2], x1 = f.v[p][e >> 1][(e & 1) * 2 + 1];
                uint32_t a, b, c;
                if (cut) {
                    const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
                    a = __builtin_amdgcn_perm(u1, u0, 0x07060302);
                    rest |= u0 | u1;
                    if (WAY == REST) gs_split_rest(x0 - __uint_as_float(u0 & 0xffff0000u), x1 - __uint_as_float(u1 & 0xffff0000u), b, c, lost[p]);
                } else {
                    gs_split(x0, x1, a, b, c, lost[p]);
                }
                hi[e] = a;
                if (!cut || WAY == REST) { mid[e] = b; lo[e] = c; }
            }
            *reinterpret_cast<gs_u32x4_t*>(to + dst[p]) = hi;
            if (!cut || WAY == REST) {
                *reinterpret_cast<gs_u32x4_t*>(to + dst[p] + PLANE) = mid;
                *reinterpret_cast<gs_u32x4_t*>(to + dst[p] + 2 * PLANE) = lo;
            }
        }
    };
    constexpr bool FOLD = NT * MT == 1;
    gs_f32x16_t big[NT][MT], small[NT][MT], sum;
    auto products = [&](int s, auto way) __attribute__((always_inline)) {
        constexpr int WAY = decltype(way)::value;
        const char* from = lds + (s & 1) * STAGE + h * GS_PIECE + i * 16;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            gs_bf16x8_t a[MT][3], w[NT][3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int m = 0; m < MT; ++m) a[m][q] = *reinterpret_cast<const gs_bf16x8_t*>(from + (wm * MT + m) * GS_GROUP + ks * 2 * GS_PIECE + q * PLANE);
#pragma unroll
                for (int n = 0; n < NT && (q == 0 ? WAY != REST : WAY != WHOLE); ++n) w[n][q] = *reinterpret_cast<const gs_bf16x8_t*>(from + (BM / 32 + wn * NT + n) * GS_GROUP + ks * 2 * GS_PIECE + q * PLANE);
            }
#define GS_MFMA(SUM, WQ, AQ)                                                                                                     \
    _Pragma("unroll") for (int n = 0; n < NT; ++n) _Pragma("unroll") for (int m = 0; m < MT; ++m)                                \
        SUM[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[n][WQ], a[m][AQ], SUM[n][m], 0, 0, 0);
            if constexpr (WAY != REST) {
                GS_MFMA(big, 0, 0)
                GS_MFMA(small, 0, 1)
            }
            if constexpr (WAY != WHOLE) {
                GS_MFMA(small, 1, 0)
                GS_MFMA(small, 1, 1)
            }
            if constexpr (WAY != REST) {
                GS_MFMA(small, 0, 2)
            } else {
                GS_MFMA(small, 1, 2)
            }
            if constexpr (WAY != WHOLE) {
                GS_MFMA(small, 2, 0)
            }
        }
    };
    // The sums of steps 0 .. steps - 1 from step0 on, the first four of which are in f0 .. f3.  Step s runs from LDS stage s & 1; behind it the pieces
    // of step s + 1 are split into the other one.  Returns the steps done: WHOLE looks at `rest` behind its first stage, behind every eighth
    // and behind its last, and ends where any of it is set.  (no_bf16 is set by the barrier that it is read behind, and is never taken back.)
    Pieces f0, f1, f2, f3;
    int done = 0;
    auto note = [&]() __attribute__((always_inline)) { if (__any((rest & 0xffffu) != 0)) no_bf16 = 1; };
    auto noted = [&]() { return __builtin_amdgcn_readfirstlane(no_bf16) != 0; };
    auto run = [&](auto way) __attribute__((always_inline)) {
        constexpr bool LOOK = decltype(way)::value == WHOLE;
        stage(f0, 0, way);
        if (LOOK) note();
        __syncthreads();
        if (LOOK && noted()) return 0;
        int s = 0;
#define GS_STEP(FREE, NEXT, S, LOOKS)     \
    fetch(FREE, (S) + 4);                 \
    products(S, way);                     \
    stage(NEXT, (S) + 1, way);            \
    __builtin_amdgcn_sched_barrier(0);    \
    if (LOOKS) note();                    \
    __syncthreads();
        for (; s + 4 < steps; s += 4) {
            const bool looks = LOOK && (s & 4);
            GS_STEP(f0, f1, s, false)
            GS_STEP(f1, f2, s + 1, false)
            GS_STEP(f2, f3, s + 2, false)
            GS_STEP(f3, f0, s + 3, looks)
            if (FOLD && ((s + done) & 28) == 28) {                 // (`done` is a multiple of eight)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    sum[e] += big[0][0][e];
                    big[0][0][e] = 0.f;
                }
            }
            if (looks && noted()) return s + 4;
        }
#undef GS_STEP
        products(s, way);
#define GS_LAST(NEXT, S)        \
    if ((S) < steps) {          \
        stage(NEXT, S, way);    \
        __syncthreads();        \
        products(S, way);       \
    }
        GS_LAST(f1, s + 1)
        GS_LAST(f2, s + 2)
        GS_LAST(f3, s + 3)
#undef GS_LAST
        if (LOOK) {
            note();
            __syncthreads();
        }
        return steps;
    };
    auto fetch_first = [&]() __attribute__((always_inline)) {
        fetch(f0, 0);
        fetch(f1, 1);
        fetch(f2, 2);
        fetch(f3, 3);
    };
    fetch_first();
    if (tid == 0) no_bf16 = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) sum[e] = 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 16; ++e) big[n][m][e] = small[n][m][e] = 0.f;
    __syncthreads();
    const int whole_steps = run(std::integral_constant<int, WHOLE>{});
    if (noted()) {
        // what the steps since the last look left out, and the others in full
        const int all = steps;
        if (whole_steps > 0) {
            done = max(0, (whole_steps - 1) & ~7);
            step0 = part0 + done;
            steps = whole_steps - done;
            fetch_first();
            run(std::integral_constant<int, REST>{});
            __syncthreads();
        }
        done = whole_steps;
        step0 = part0 + done;
        steps = all - done;
        if (steps > 0) {
            if (done > 0) fetch_first();
            run(std::integral_constant<int, FULL>{});
        }
    }
    // Two kinds of values do not split, and the sums that they are in are formed once more by float32 instructions, the wave's other values
    // stay: those beyond bfloat16's range, infinities and NaN, whose rest is a NaN as every sum with it then, and those below 2^-110 or so, of
    // which bits are lost: their rows of A and W
    uint32_t again[NT][MT];
    bool any = false;
    uint32_t short_of = 0;
#pragma unroll
    for (int p = 0; p < P; ++p) short_of |= lost[p];
    const bool shorts = __syncthreads_or((short_of & 0xffffu) != 0);                // (and the stages are free)
    uint32_t* row_lost = reinterpret_cast<uint32_t*>(lds);                          // [BM + BN][4]
    if (shorts) {
#pragma unroll
        for (int p = 0; p < P; ++p) row_lost[(sr + p * ROWS) * 4 + kp] = lost[p] & 0xffffu;
        __syncthreads();
    }
    auto lost_in = [&](int row) { const gs_u32x4_t f = *reinterpret_cast<const gs_u32x4_t*>(row_lost + row * 4); return (f[0] | f[1] | f[2] | f[3]) != 0; };
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            again[n][m] = 0;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                big[n][m][e] += FOLD ? small[n][m][e] + sum[e] : small[n][m][e];
                again[n][m] |= fabsf(big[n][m][e]) < INFINITY ? 0u : 1u << e;
            }
            if (shorts) {
                if (lost_in((wm * MT + m) * 32 + i)) again[n][m] = 0xffffu;
                for (int e = 0; e < 16; ++e)
                    if (lost_in(BM + (wn * NT + n) * 32 + 8 * (e >> 2) + 4 * h + (e & 3))) again[n][m] |= 1u << e;
            }
            any |= again[n][m] != 0;
        }
    if (__any(any)) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float* a_at = A + (size_t)min(m0 + (wm * MT + m) * 32 + i, M - 1) * K + 4 * h;
                const float* w_at = W + (size_t)w_row((wn * NT + n) * 32 + i) * K + 4 * h;
                gs_f32x16_t total, acc;
#pragma unroll
                for (int e = 0; e < 16; ++e) total[e] = acc[e] = 0.f;
                const int end = part1 * GS_BK;
                for (int k0 = part0 * GS_BK; k0 < end; k0 += 256) {                // a chain ends every 256 of K, as in gemm_f32.hip
#pragma unroll 4
                    for (int k = k0; k < min(k0 + 256, end); k += 8) {
                        const gs_f32x4_t va = *reinterpret_cast<const gs_f32x4_t*>(a_at + k), vw = *reinterpret_cast<const gs_f32x4_t*>(w_at + k);
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(vw[j], va[j], acc, 0, 0, 0);
                    }
#pragma unroll
                    for (int e = 0; e < 16; ++e) { total[e] += acc[e]; acc[e] = 0.f; }
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) big[n][m][e] = again[n][m] >> e & 1 ? total[e] : big[n][m][e];
            }
    }
    // lane (i, h) has C[row i][columns 8 q + 4 h .. + 3], q < 4; GATED: gate values at q < 2, the same columns' up values at q + 2
    const int width = GATED ? N / 2 : N;
    const bool whole = (width & 3) == 0;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = m0 + (wm * MT + m) * 32 + i;
        if (row >= M) continue;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int q = 0; q < (GATED ? 2 : 4); ++q) {
                const int col = (GATED ? n0 / 2 + (wn * NT + n) * 16 : n0 + (wn * NT + n) * 32) + 8 * q + 4 * h;
                float* to = C + (size_t)row * width + col;
                gs_f32x4_t y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = GATED ? gated_value(act, big[n][m][4 * q + e], big[n][m][4 * (q + 2) % 16 + e]) : big[n][m][4 * q + e];
                if (whole) {
                    if (col < width) *reinterpret_cast<gs_f32x4_t*>(to) = y;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < width) to[e] = y[e];
                }
            }
    }
}

// ---- dispatch --------------------------------------------------------------------------------------------------------------
// Estimated time of both tiles for a matrix of float32 values, fitted to 120 launches of 40 to 611 rows, K of 1024 to 6144 and 1 to 12 parts:
// a compute unit takes 0.9 us for a step of a large block (1.03 with the chip full), 0.5 us for one small block, 0.83 for two, 1.0 with the
// chip full.  A widened matrix takes two thirds of it with either tile, so that the choice is the same: over 344 launches of 38 to 1435 rows it is 0.5 %
// behind the better tile for float32 values, 0.4 % for widened ones (17 and 13 % at most, in 12 parts).  Large / small tile, us, float32 values and
// widened: 611 rows, 4096 x 1024 (160 or 640 blocks) 40.5 / 49.1 and 29.8 / 35.9, 1024 x 2048 in three parts 28.7 / 25.5 and 21.7 / 18.2, 400
// rows, 4096 x 2048 71.4 / 63.4 and 51.5 / 44.9, 12288 x 2048 160 / 178 and 110 / 122.  A chain of products of the large tile is the part's whole
// K, which to 2048 rounds no more than the float32 instructions do; the small tile's sums change every 1024.
static bool gs_large_tile(int M, int N, int K, int parts) {
    const int64_t large = (int64_t)((M + 127) / 128) * ((N + 127) / 128) * parts, small = (int64_t)((M + 63) / 64) * ((N + 63) / 64) * parts;
    const double steps = (double)K / GS_BK / parts, rest = small % 512 == 0 ? 0.0 : (small % 512 <= 256 ? 0.5 : 0.83);
    return K / parts <= 2048
        && 8.0 + steps * (double)((large + 255) / 256) * (0.9 + 0.13 * (large < 256 ? large / 256.0 : 1.0)) <= 5.0 + steps * ((double)(small / 512) + rest);
}

// More than 32 rows (below, the products are bound by W's way from memory: 24 rows, 4096 x 1024 8.7 us / 18.7), and without parts tiles
// for half of the compute units (2048 x 2048, 90 rows: 64 tiles 22 / 33; 4096 x 2048: 128 tiles 38.5 / 30.5 with a widened matrix, 38.3 with one of
// float32 values; the smallest of that many, 4096 x 1024, 22.8 / 18.0 and 22.5; 65 rows, the fewest of two tiles, 36.1 / 30.3 and 38.2, 20.9 / 17.8 and
// 21.9: what float32 values lose there is less than widened ones, which a call cannot tell from them beforehand, gain).
bool gemm_f32_split_takes(int M, int N, int K, int parts) {
    return M > 32 && K % GS_BK == 0 && (int64_t)M * K < (1 << 29) && (int64_t)N * K < (1 << 29)
        && (parts > 1 || (int64_t)((M + 63) / 64) * ((N + 63) / 64) >= 128);
}

template <int BM, int BN, int WM, int WN, bool GATED>
static int gs_launch(const float* A, const float* W, float* C, int M, int N, int K, int parts, GateAct act, hipStream_t st) {
    const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    const int64_t blocks = (int64_t)tm * tn * parts;
    SPY_REQUIRE(parts >= 1 && parts <= K / GS_BK && blocks < (1 << 28), "spy_gemm (float32): %d parts of %d x %d x %d", parts, M, N, K);
    gemm_f32_split_kernel<BM, BN, WM, WN, GATED><<<(unsigned)((blocks + 7) / 8 * 8), 64 * WM * WN, 0, st>>>(A, W, C, M, N, K, tm, tn, parts, act);
    SPY_CHECK_LAUNCH("spy_gemm (float32)");
    return 0;
}

int gemm_f32_split(const float* A, const float* W, float* C, int M, int N, int K, int parts, hipStream_t st) {
    const GateAct none = {1.f, 0.f};
    return gs_large_tile(M, N, K, parts) ? gs_launch<128, 128, 2, 4, false>(A, W, C, M, N, K, parts, none, st)
                                         : gs_launch<64, 64, 2, 2, false>(A, W, C, M, N, K, parts, none, st);
}

int gemm_f32_split_gated(const float* A, const float* W, float* C, int M, int N, int K, GateAct act, hipStream_t st) {
    return gs_large_tile(M, N, K, 1) ? gs_launch<128, 128, 2, 4, true>(A, W, C, M, N, K, 1, act, st)
                                     : gs_launch<64, 64, 2, 2, true>(A, W, C, M, N, K, 1, act, st);
}
