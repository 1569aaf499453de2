// Mixture of experts: the router's choice, the (token, choice) pairs sorted by expert, the experts' products over the
// sorted rows, and the weighted sum of a token's results.  Nothing here needs the host to know how many tokens an
// expert got: the sizes of all arrays follow the number of tokens alone, and blocks whose tile holds no rows leave.
//
//   route:   s = softmax(z) over all experts (float32); choice = s + correction; the experts form `groups` equal runs of
//            neighbours, a group's score is its largest choice, only experts of the `keep` best groups can be chosen (the
//            others count as minus infinity); the `top` largest choices are taken; their weights are s (without the
//            correction) over their sum (+ 1e-20), times `scale`.
//   align:   rows of the sorted order: expert e's pairs in a run that starts at a multiple of MOE_TM rows, padded with -1.
//   gemm:    C[row] = A[source of row] . W[expert of the row's tile]^T, float32 products and sums; optionally gated:
//            W = [gate rows | up rows], C = silu(gate) * up; or (MoeAct kind 1) with the row's weight w multiplied into both
//            sums first, g = min(w gate, limit), u = clamp(w up, -limit, limit), C = g sigmoid(1.702 g) (u + 1).
//            Experts without a gate: W = [up rows], C = gelu(up).
//            Where tables name the experts by token id, the align step of all mixtures is one launch ahead of the layers.
//   combine: out[t] = scale * sum_k weight[t, k] * Y[row of pair (t, k)].
#include "gemm_rows.h"
#include <math.h>
#include <type_traits>

#define MOE_TM 16
#define MOE_MAX_EXPERTS 1024

// What a gated product does with its two sums (see the top), and one without a gate with its sum: kind 2: gelu (exact); else
// nothing.  pair_w: the weight of every (token, choice) pair, or null.
struct MoeAct {
    int kind;
    float limit;
    const float* pair_w;
};
__device__ __forceinline__ float moe_gated(float g, float u, const MoeAct& a, float w) {
    if (a.kind == 0) return g / (1.0f + expf(-g)) * u;
    g = fminf(g * w, a.limit);
    u = fminf(fmaxf(u * w, -a.limit), a.limit);
    return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
}
__device__ __forceinline__ float moe_ungated(float v, const MoeAct& a) { return a.kind == 2 ? gelu_f(v) : v; }

// one wave per token
__global__ __launch_bounds__(64) void moe_route_kernel(int* __restrict__ ids, float* __restrict__ weights, const float* __restrict__ z,
                                                       const float* __restrict__ correction, int E, int top, int groups, int keep,
                                                       float scale, int sigmoid, int renorm, const float* __restrict__ zbias) {
    // zbias != null: a bias [E] that is part of the logits (it moves the scores and with them the weights, where the
    // correction moves the choice alone)
    __shared__ float sc[MOE_MAX_EXPERTS], ch[MOE_MAX_EXPERTS], gsc[MOE_MAX_EXPERTS];
    __shared__ float zb[MOE_MAX_EXPERTS];
    __shared__ int allowed[MOE_MAX_EXPERTS], sel[MOE_MAX_EXPERTS];
    const int t = blockIdx.x, lane = threadIdx.x;
    const float* zr = z + (size_t)t * E;
    if (zbias) {
        for (int e = lane; e < E; e += 64) zb[e] = zr[e] + zbias[e];     // (a lane reads back only what it wrote: no barrier)
        zr = zb;
    }
    if (sigmoid) {
        // every logit by itself
        for (int e = lane; e < E; e += 64) {
            sc[e] = 1.0f / (1.0f + expf(-zr[e]));
            ch[e] = sc[e] + (correction ? correction[e] : 0.f);
        }
    } else {
        float mx = -INFINITY;
        for (int e = lane; e < E; e += 64) mx = fmaxf(mx, zr[e]);
        mx = wave_max(mx);
        float sum = 0.f;
        for (int e = lane; e < E; e += 64) {
            const float p = expf(zr[e] - mx);
            sc[e] = p;
            sum += p;
        }
        sum = wave_sum(sum);
        for (int e = lane; e < E; e += 64) {
            sc[e] = sc[e] / sum;
            ch[e] = sc[e] + (correction ? correction[e] : 0.f);
        }
    }
    __syncthreads();
    const int per = E / groups;
    for (int g = lane; g < groups; g += 64) {
        float best = -INFINITY;
        for (int i = 0; i < per; ++i) best = fmaxf(best, ch[g * per + i]);
        gsc[g] = best;
        allowed[g] = 0;
    }
    __syncthreads();
    for (int r = 0; r < keep; ++r) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
        for (int g = lane; g < groups; g += 64)
            if (!allowed[g] && (gsc[g] > bv || (gsc[g] == bv && g < bi))) { bv = gsc[g]; bi = g; }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (lane == 0 && bi < groups) allowed[bi] = 1;
        __syncthreads();
    }
    for (int e = lane; e < E; e += 64)
        if (!allowed[e / per]) ch[e] = -INFINITY;
    __syncthreads();
    float wsum = 0.f;
    for (int r = 0; r < top; ++r) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
        for (int e = lane; e < E; e += 64)
            if (ch[e] > bv) { bv = ch[e]; bi = e; }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (bi >= E) bi = 0;                       // fewer allowed experts than choices: never the case for a checked configuration
        wsum += sc[bi];
        __syncthreads();
        if (lane == 0) { ch[bi] = -INFINITY; sel[r] = bi; }
        __syncthreads();
    }
    const float norm = renorm ? scale / (wsum + 1e-20f) : scale;
    for (int r = lane; r < top; r += 64) {
        ids[(size_t)t * top + r] = sel[r];
        weights[(size_t)t * top + r] = sc[sel[r]] * norm;
    }
}

extern "C" int spy_moe_route(int* ids, float* weights, const float* z, const float* correction, int T, int E, int top, int groups,
                             int keep, float scale, int sigmoid, int renorm, const float* zbias, hipStream_t st) {
    SPY_REQUIRE(T > 0 && E > 0 && E <= MOE_MAX_EXPERTS, "spy_moe_route: %d experts (1..%d)", E, MOE_MAX_EXPERTS);
    SPY_REQUIRE(groups > 0 && E % groups == 0 && keep > 0 && keep <= groups && top > 0 && top <= keep * (E / groups),
                "spy_moe_route: %d of %d groups of %d experts cannot give %d choices", keep, groups, E / (groups > 0 ? groups : 1), top);
    moe_route_kernel<<<T, 64, 0, st>>>(ids, weights, z, correction, E, top, groups, keep, scale, sigmoid, renorm, zbias);
    SPY_CHECK_LAUNCH("spy_moe_route");
    return 0;
}

// Groups of neighbouring row tiles of one expert, which the products of many rows per expert go by: [0] how many there are, then two
// ints for each: first tile * 16 + tiles (MOE_GROUP of them but for an expert's last group), and its band, first group * 8 + groups:
// up to MOE_BAND groups of one expert whose blocks run beside each other.
#define MOE_GROUP 8
#define MOE_BAND 4
__device__ __host__ __forceinline__ int moe_max_groups(int max_tiles, int E, int P) { return max_tiles / MOE_GROUP + (E < P ? E : P); }

// One block.  Pair p's expert is expert_of(p) (outside 0 .. E - 1: the pair has no row) -> sorted_pair [max_tiles MOE_TM]
// (pair or -1), pair_row [P], tile_expert [max_tiles] (expert or -1), group [1 + 2 moe_max_groups].
template <typename F>
__device__ __forceinline__ void moe_align_block(int* __restrict__ sorted_pair, int* __restrict__ pair_row, int* __restrict__ tile_expert,
                                                int* __restrict__ group, F expert_of, int P, int E, int max_tiles) {
    __shared__ int count[MOE_MAX_EXPERTS], first[MOE_MAX_EXPERTS], cursor[MOE_MAX_EXPERTS], first_group[MOE_MAX_EXPERTS];
    __shared__ int total_tiles;
    const int tid = threadIdx.x;
    for (int e = tid; e < E; e += blockDim.x) { count[e] = 0; cursor[e] = 0; }
    __syncthreads();
    for (int p = tid; p < P; p += blockDim.x) {
        const int e = expert_of(p);
        if (e >= 0 && e < E) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (tid == 0) {
        int tiles = 0, groups = 0;
        for (int e = 0; e < E; ++e) {
            const int nt = (count[e] + MOE_TM - 1) / MOE_TM;
            first[e] = tiles;
            first_group[e] = groups;
            tiles += nt;
            groups += (nt + MOE_GROUP - 1) / MOE_GROUP;
        }
        total_tiles = tiles;
        group[0] = min(groups, moe_max_groups(max_tiles, E, P));
    }
    __syncthreads();
    for (int e = tid; e < E; e += blockDim.x) {
        const int nt = (count[e] + MOE_TM - 1) / MOE_TM;
        for (int i = 0; i < nt && first[e] + i < max_tiles; ++i) tile_expert[first[e] + i] = e;
        for (int i = 0; i * MOE_GROUP < nt && first_group[e] + i < moe_max_groups(max_tiles, E, P); ++i)
        {
            const int ng = (nt + MOE_GROUP - 1) / MOE_GROUP, band = i / MOE_BAND * MOE_BAND, at = 1 + 2 * (first_group[e] + i);
            group[at] = (first[e] + i * MOE_GROUP) * 16 + min(MOE_GROUP, nt - i * MOE_GROUP);
            group[at + 1] = (first_group[e] + band) * 8 + min(MOE_BAND, ng - band);
        }
        for (int r = count[e]; r < nt * MOE_TM; ++r)
            if (first[e] * MOE_TM + r < max_tiles * MOE_TM) sorted_pair[first[e] * MOE_TM + r] = -1;
    }
    for (int i = total_tiles + tid; i < max_tiles; i += blockDim.x) tile_expert[i] = -1;
    for (int r = total_tiles * MOE_TM + tid; r < max_tiles * MOE_TM; r += blockDim.x) sorted_pair[r] = -1;
    for (int p = tid; p < P; p += blockDim.x) {
        const int e = expert_of(p);
        if (e < 0 || e >= E) { pair_row[p] = -1; continue; }
        const int row = first[e] * MOE_TM + atomicAdd(&cursor[e], 1);
        if (row < max_tiles * MOE_TM) sorted_pair[row] = p;
        pair_row[p] = row < max_tiles * MOE_TM ? row : -1;
    }
}

__global__ __launch_bounds__(1024) void moe_align_kernel(int* __restrict__ sorted_pair, int* __restrict__ pair_row,
                                                         int* __restrict__ tile_expert, int* __restrict__ group,
                                                         const int* __restrict__ ids, int P, int E, int max_tiles) {
    moe_align_block(sorted_pair, pair_row, tile_expert, group, [=](int p) { return ids[p]; }, P, E, max_tiles);
}

// Experts named by tables of the token ids: all of a step's mixtures at once, one block per mixture.  Mixture l: the table
// [V, top] (int32), E experts; pair p = (token p / top, choice p % top).  out: the mixtures' arrays one after the other, each
// sorted_pair [max_tiles MOE_TM], pair_row [T top], tile_expert [max_tiles], group [1 + 2 moe_max_groups], every array rounded up to
// four ints.
struct MoeTable { const int* table; int E, top; };
__device__ __forceinline__ int moe_up4(int n) { return (n + 3) & ~3; }
__global__ __launch_bounds__(1024) void moe_align_tables_kernel(int* __restrict__ out, const MoeTable* __restrict__ tables,
                                                                const int* __restrict__ ids, int T, int V) {
    size_t off = 0;
    int P = 0, max_tiles = 0, groups = 0;
    for (int l = 0; l <= (int)blockIdx.x; ++l) {
        if (l) off += moe_up4(max_tiles * MOE_TM) + moe_up4(P) + moe_up4(max_tiles) + moe_up4(1 + 2 * groups);
        P = T * tables[l].top;
        max_tiles = P / MOE_TM + min(tables[l].E, P);
        groups = moe_max_groups(max_tiles, tables[l].E, P);
    }
    const MoeTable tb = tables[blockIdx.x];
    int* sorted_pair = out + off;
    int* pair_row = sorted_pair + moe_up4(max_tiles * MOE_TM);
    int* tile_expert = pair_row + moe_up4(P);
    int* group = tile_expert + moe_up4(max_tiles);
    const int top = tb.top;
    const int* table = tb.table;
    moe_align_block(sorted_pair, pair_row, tile_expert, group, [=](int p) {
        const int t = p / top, id = ids[t];
        return id >= 0 && id < V ? table[(size_t)id * top + (p - t * top)] : -1;
    }, P, tb.E, max_tiles);
}

// tables: MoeTable [n] on the device; max_experts, max_top: the largest E and top among them (the caller's account of what the
// device array holds).
extern "C" int spy_moe_align_tables(int* out, int64_t out_ints, const void* tables, int n, int max_experts, int max_top, const int* ids,
                                    int T, int V, hipStream_t st) {
    SPY_REQUIRE(n > 0 && n <= 65535 && T > 0 && V > 0 && max_experts > 0 && max_experts <= MOE_MAX_EXPERTS && max_top > 0,
                "spy_moe_align_tables: %d tables of up to %d experts (1..%d)", n, max_experts, MOE_MAX_EXPERTS);
    SPY_REQUIRE((int64_t)T * max_top <= (1 << 26), "spy_moe_align_tables: too many (token, choice) pairs");
    SPY_REQUIRE(out && out_ints > 0 && ((uintptr_t)tables % 8) == 0, "spy_moe_align_tables: no output");
    moe_align_tables_kernel<<<n, 1024, 0, st>>>(out, (const MoeTable*)tables, ids, T, V);
    SPY_CHECK_LAUNCH("spy_moe_align_tables");
    return 0;
}

extern "C" int spy_moe_align(int* sorted_pair, int* pair_row, int* tile_expert, int* group, const int* ids, int P, int E, int max_tiles,
                             hipStream_t st) {
    SPY_REQUIRE(P > 0 && E > 0 && E <= MOE_MAX_EXPERTS, "spy_moe_align: %d experts (1..%d)", E, MOE_MAX_EXPERTS);
    SPY_REQUIRE(max_tiles >= P / MOE_TM + (E < P ? E : P), "spy_moe_align: %d tiles are too few for %d pairs of %d experts", max_tiles, P, E);
    moe_align_kernel<<<1, 1024, 0, st>>>(sorted_pair, pair_row, tile_expert, group, ids, P, E, max_tiles);
    SPY_CHECK_LAUNCH("spy_moe_align");
    return 0;
}

extern "C" int spy_moe_tile_rows() { return MOE_TM; }
extern "C" int spy_moe_group_ints(int max_tiles, int E, int P) { return 1 + 2 * moe_max_groups(max_tiles, E, P); }

// A tile of MOE_TM sorted rows x 64 columns per block; 256 threads, thread (ty, tx) has row ty and columns 4 tx .. + 3.
// gather > 0: row r reads A[sorted_pair[r] / gather] (the token of the pair); 0: A[r].  TILED: the experts' matrices lie in operand
// order (gemm_decode.h), where four neighbours in K are neighbours too: float32 rows of matrices that are kept so for bfloat16 ones.
// Measured, both products of 32 experts of 2 x 1536 x 2048, four a token, us, matrices in row order / in operand order with a copy in row
// order made in every call / as they lie: 4 tokens 483 / 1038 / 392, 200 tokens 1108 / 1615 / 731.
#define MG_TN 64
#define MG_K 16
template <typename TA, typename TW, typename TC, bool GATED, bool TILED>
__global__ __launch_bounds__(256) void moe_gemm_kernel(TC* __restrict__ C, const TA* __restrict__ A, const TW* __restrict__ W,
                                                       const int* __restrict__ tile_expert, const int* __restrict__ sorted_pair,
                                                       int gather, int N, int K, long long w_stride, MoeAct act) {
    __shared__ float As[MG_K][MOE_TM + 1];
    __shared__ float Ws[GATED ? 2 : 1][MG_K][MG_TN + 4];
    __shared__ int src[MOE_TM];
    const int tile = blockIdx.y;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int n0 = blockIdx.x * MG_TN;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    if (threadIdx.x < MOE_TM) {
        const int p = sorted_pair[tile * MOE_TM + threadIdx.x];
        src[threadIdx.x] = p < 0 ? -1 : (gather > 0 ? p / gather : tile * MOE_TM + (int)threadIdx.x);
    }
    __syncthreads();
    const TW* We = W + (size_t)e * w_stride;
    float acc[4] = {}, acc2[4] = {};
    // staging: A 16 x 16 values, one per thread; W 64 x 16 values, four per thread
    const int ar = threadIdx.x >> 4, ak = threadIdx.x & 15;
    const int wr = threadIdx.x >> 2, wk = (threadIdx.x & 3) * 4;
    const int w_tiles = (GATED ? 2 : 1) * N / 16;
    auto w_at = [&](int n, int k) {
        if (!TILED) return (size_t)n * K + k;
        return ((size_t)(k >> 7) * w_tiles + (n >> 4)) * 2048 + ((k >> 5) & 3) * 512 + ((k >> 3) & 3) * 128 + (n & 15) * 8 + (k & 7);
    };
    for (int k0 = 0; k0 < K; k0 += MG_K) {
        {
            const int sr = src[ar], k = k0 + ak;
            As[ak][ar] = (sr >= 0 && k < K) ? to_f32<TA>(A[(size_t)sr * K + k]) : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = k0 + wk + i, n = n0 + wr;
            Ws[0][wk + i][wr] = (n < N && k < K) ? to_f32<TW>(We[w_at(n, k)]) : 0.f;
            if (GATED) Ws[GATED ? 1 : 0][wk + i][wr] = (n < N && k < K) ? to_f32<TW>(We[w_at(N + n, k)]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < MG_K; ++k) {
            const float a = As[k][ty];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[i] = fmaf(a, Ws[0][k][tx * 4 + i], acc[i]);
                if (GATED) acc2[i] = fmaf(a, Ws[GATED ? 1 : 0][k][tx * 4 + i], acc2[i]);
            }
        }
        __syncthreads();
    }
    if (src[ty] < 0) return;
    const size_t row = (size_t)tile * MOE_TM + ty;
    const float rw = (GATED && act.pair_w) ? act.pair_w[sorted_pair[row]] : 1.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + tx * 4 + i;
        if (n >= N) continue;
        float v = acc[i];
        if (GATED) {
            v = moe_gated(acc[i], acc2[i], act, rw);
        } else {
            v = moe_ungated(v, act);
        }
        C[row * N + n] = from_f32<TC>(v);
    }
}


// The same product on the matrix cores, bfloat16 operands and float32 sums (v_mfma_f32_16x16x32_bf16), for few rows per expert (decoding)
// and for experts so few or small that blocks of 128 rows would leave the chip idle (ops.experts_by_groups has the line):
// a block has one row tile (16 sorted rows) and 32 rows of W (gated: 16 gate rows and the 16 up rows of the same columns), whose K
// its four waves take in chunks of 128 in turn and add through LDS.  Operands go from memory straight into MFMA operand registers: lane
// (r = lane % 16, g = lane / 16) holds row r, values k + 8 g .. + 7; the result tile is C^T: lane (r, g) holds C[row r][column 4 g + i].
// What bounds it: the experts' matrices from memory.  A wave that walks all of K for 32 rows of W has four times the work of one that
// takes a quarter, and the last round of such blocks, a sixth of the chip, costs what a whole one does.  Measured, both products of 32
// experts of 2 x 3072 x 4096, 12 tokens with four each: 199 + 105 us (6.4 TB/s over the experts touched) against 236 + 141 for such
// blocks; 8 tokens, 2 x 1536 x 2048: 43 + 20 against 60 + 42.  Blocks of one expert's columns are neighbours in the grid (229 + 123 us
// with an expert's tiles outermost); loads with the hint that they are not read again cost a fifth (245 + 134): a row's 64 bytes of
// one load are half a line, the other half is the next load's.
typedef __attribute__((__vector_size__(8 * sizeof(short)))) short moe_bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float moe_f32x4_t;

// TILED: the experts' matrices lie in operand order (gemm_decode.h), so that a load is 1 KB in one piece.
template <bool GATED, bool TILED, typename TC>
__global__ __launch_bounds__(256) void moe_gemm_tile_kernel(TC* __restrict__ C, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                            const int* __restrict__ tile_expert, const int* __restrict__ sorted_pair,
                                                            int gather, int N, int K, long long w_stride, MoeAct act) {
    __shared__ __align__(16) float red[4][2][64][4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int t = blockIdx.y, n0 = blockIdx.x * (GATED ? 16 : 32);
    const int e = __builtin_amdgcn_readfirstlane(tile_expert[t]);
    if (e < 0) return;
    const int row = t * MOE_TM + r, p = sorted_pair[row], p0 = sorted_pair[t * MOE_TM];
    // a tile with an expert has a first row; rows that do not exist read that one's values, and what they give is not stored
    const int src = gather > 0 ? max(p >= 0 ? p : p0, 0) / gather : (p >= 0 ? row : t * MOE_TM);
    const bf16_t* xrow = A + (size_t)src * K + 8 * g;
    const bf16_t* We = W + (size_t)e * w_stride;
    const bf16_t* wrow[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        if (TILED) wrow[nt] = We + (size_t)(GATED ? (nt * N + n0) / 16 : min(n0 / 16 + nt, N / 16 - 1)) * 2048 + lane * 8;
        else wrow[nt] = We + (size_t)(GATED ? nt * N + min(n0 + r, N - 1) : min(n0 + nt * 16 + r, N - 1)) * K + 8 * g;
    }
    const size_t w_step = TILED ? 512 : 32, w_wide = TILED ? (size_t)(GATED ? 2 : 1) * N : 1;          // (a chunk's values are K's 128 of all rows)
    moe_f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    auto load = [&](const bf16_t* q) { return *reinterpret_cast<const moe_bf16x8_t*>(q); };
    auto fetch = [&](moe_bf16x8_t (&a)[2][4], moe_bf16x8_t (&b)[4], int k) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) a[nt][j] = load(wrow[nt] + k * w_wide + w_step * j);
            b[j] = *reinterpret_cast<const moe_bf16x8_t*>(xrow + k + 32 * j);
        }
    };
    auto products = [&](const moe_bf16x8_t (&a)[2][4], const moe_bf16x8_t (&b)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[nt][j], b[j], acc[nt], 0, 0, 0);
    };
    // two sets of operands taken in turn, the next chunk's asked for ahead of this one's products (no load under a condition)
    const int chunks = K >> 7, mine = (chunks - wave + 3) >> 2;
    moe_bf16x8_t a0[2][4], b0[4], a1[2][4], b1[4];
    if (mine > 0) {
        auto at = [&](int i) { return (wave + 4 * i) << 7; };
        fetch(a0, b0, at(0));
        int i = 0;
        for (; i + 2 < mine; i += 2) {
            fetch(a1, b1, at(i + 1));
            products(a0, b0);
            fetch(a0, b0, at(i + 2));
            products(a1, b1);
        }
        if (i + 1 < mine) {
            fetch(a1, b1, at(i + 1));
            products(a0, b0);
            products(a1, b1);
        } else {
            products(a0, b0);
        }
    }
    if (!TILED && wave == (chunks & 3)) {                    // the rest of K (a multiple of 8): the wave whose turn it would be
        const moe_bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int k = chunks << 7; k < K; k += 32) {
            const bool kok = k + 8 * g < K;
            const moe_bf16x8_t b = kok ? *reinterpret_cast<const moe_bf16x8_t*>(xrow + k) : zero8;
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                const moe_bf16x8_t a = kok ? load(wrow[nt] + k) : zero8;
                acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[nt], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) *reinterpret_cast<moe_f32x4_t*>(red[wave][nt][lane]) = acc[nt];
    __syncthreads();
    if (wave > (GATED ? 0 : 1) || p < 0) return;
    moe_f32x4_t sum[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        sum[nt] = *reinterpret_cast<const moe_f32x4_t*>(red[0][nt][lane]);
#pragma unroll
        for (int w = 1; w < 4; ++w) sum[nt] += *reinterpret_cast<const moe_f32x4_t*>(red[w][nt][lane]);
    }
    if (GATED) {
        const float rw = act.pair_w ? act.pair_w[p] : 1.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = n0 + 4 * g + i;
            if (col < N) C[(size_t)row * N + col] = from_f32<TC>(moe_gated(sum[0][i], sum[1][i], act, rw));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = n0 + wave * 16 + 4 * g + i;
            if (col < N) C[(size_t)row * N + col] = from_f32<TC>(moe_ungated(wave ? sum[1][i] : sum[0][i], act));
        }
    }
}


// Many rows per expert: the same tiles, but the gathered rows of A go through LDS once per block and step of 128 of K
// (the four waves read the same rows; loaded by each of them they swept the first-level cache), while every wave's W
// fragments still come straight from memory, asked for before the block waits for the staged rows.
#define MOE_ROWS 128                 // 8 row tiles
#define MOE_DIES 8
#define MOE_LDS_STRIDE (128 + 8)     // values per staged row (16-byte pieces; the pad spreads the rows over the banks)
template <bool GATED, typename TC>
__global__ __launch_bounds__(256, 2) void moe_gemm_mfma_lds_kernel(TC* __restrict__ C, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                const int* __restrict__ tile_expert, const int* __restrict__ sorted_pair,
                                                                int gather, int max_tiles, int N, int K, long long w_stride, MoeAct act) {
    constexpr int MT = 8, NT = 2;
    __shared__ __align__(16) bf16_t xs[MOE_ROWS * MOE_LDS_STRIDE];
    __shared__ int src_row[MOE_ROWS];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    // Blocks go to the chip's 8 dies in turn, by their number in the grid, and each die has an L2 of its own: the numbers are
    // dealt out again, so that a die gets a run of blocks in (row tiles, columns) order.  Those at work on it at one time are
    // then all columns of a few row tiles, of one or two experts, and a step's rows and matrix parts come from memory once
    // for all of them.
    int bx, by;
    {
        const int gx = gridDim.x, gy = gridDim.y, n = gx * gy, lin = blockIdx.x + gx * blockIdx.y;
        const int die = lin % MOE_DIES, idx = lin / MOE_DIES, per = (n + MOE_DIES - 1) / MOE_DIES, rem = n % MOE_DIES;
        const int v = (rem == 0 || die < rem) ? die * per + idx : rem * per + (die - rem) * (per - 1) + idx;
        bx = v / gy;
        by = v - bx * gy;
    }
    const int n0 = (by * 4 + wave) * (GATED ? 16 : 32);
    const bool cols = n0 < N;                        // (a wave without columns still helps to stage)
    int t = bx * MT;
    const int t_end = min(t + MT, max_tiles);
    const moe_bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    const int srow = threadIdx.x >> 4, spiece = threadIdx.x & 15;      // staging: rows srow + 16 i, 16-byte piece spiece
    while (t < t_end) {
        const int e = __builtin_amdgcn_readfirstlane(tile_expert[t]);
        if (e < 0) break;
        int run = 1;
        while (t + run < t_end && __builtin_amdgcn_readfirstlane(tile_expert[t + run]) == e) ++run;
        __syncthreads();                             // the run before has read its rows
        if (threadIdx.x < MOE_ROWS) {
            int src = -1;
            if ((int)threadIdx.x < run * MOE_TM) {
                const int row = t * MOE_TM + threadIdx.x;
                const int p = sorted_pair[row];
                src = p < 0 ? -1 : (gather > 0 ? p / gather : row);
            }
            src_row[threadIdx.x] = src;
        }
        __syncthreads();
        int srcs[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) srcs[i] = src_row[srow + 16 * i];
        bool xok[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xok[mt] = mt < run && src_row[mt * 16 + r] >= 0;
        const bf16_t* We = W + (size_t)e * w_stride;
        const bf16_t* wrow[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int row = GATED ? nt * N + min(n0 + r, N - 1) : min(n0 + nt * 16 + r, N - 1);
            wrow[nt] = We + (size_t)(cols ? row : 0) * K + 8 * g;
        }
        moe_f32x4_t acc[NT][MT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = moe_f32x4_t{0.f, 0.f, 0.f, 0.f};
        // the operands of a step are asked for one step ahead: W fragments into registers, the rows of A into registers
        // on their way to LDS, both in flight while the matrix cores work on the step before.  The run's tiles are walked as
        // eight, four or two: a tile that the run does not have is multiplied as it lies (its rows go nowhere), because a
        // condition around every product would make the wave wait for every operand on its own.
        moe_bf16x8_t a[NT][4], stage[MT];
#define MOE_ASK(KK)                                                                                                            \
        {                                                                                                                      \
            _Pragma("unroll") for (int j = 0; j < 4; ++j)                                                                      \
                _Pragma("unroll") for (int nt = 0; nt < NT; ++nt)                                                              \
                    a[nt][j] = (cols && (KK) + 32 * j + 8 * g < K) ? *reinterpret_cast<const moe_bf16x8_t*>(wrow[nt] + (KK) + 32 * j) : zero8; \
            const bool kin_ = (KK) + 8 * spiece < K;                                                                           \
            _Pragma("unroll") for (int i = 0; i < TILES; ++i)                                                                  \
                stage[i] = (srcs[i] >= 0 && kin_) ? *reinterpret_cast<const moe_bf16x8_t*>(A + (size_t)srcs[i] * K + (KK) + 8 * spiece) : zero8; \
        }
        auto walk = [&](auto tiles) {
            constexpr int TILES = decltype(tiles)::value;
            MOE_ASK(0)
            for (int k = 0; k < K; k += 128) {
                moe_bf16x8_t ac[NT][4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) ac[nt][j] = a[nt][j];
                __syncthreads();                     // the step before has read its rows
#pragma unroll
                for (int i = 0; i < TILES; ++i)
                    *reinterpret_cast<moe_bf16x8_t*>(xs + (srow + 16 * i) * MOE_LDS_STRIDE + 8 * spiece) = stage[i];
                __syncthreads();
                if (k + 128 < K) MOE_ASK(k + 128)
                if (cols) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int mt = 0; mt < TILES; ++mt) {
                            const moe_bf16x8_t b = *reinterpret_cast<const moe_bf16x8_t*>(xs + (mt * 16 + r) * MOE_LDS_STRIDE + 32 * j + 8 * g);
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt) acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ac[nt][j], b, acc[nt][mt], 0, 0, 0);
                        }
                }
            }
        };
        if (run > 4) walk(std::integral_constant<int, 8>{});
        else if (run > 2) walk(std::integral_constant<int, 4>{});
        else walk(std::integral_constant<int, 2>{});
#undef MOE_ASK
        if (cols) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if (mt >= run || !xok[mt]) continue;
                const size_t row = (size_t)(t + mt) * MOE_TM + r;
                if (GATED) {
                    const float rw = act.pair_w ? act.pair_w[sorted_pair[row]] : 1.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int col = n0 + 4 * g + i;
                        if (col < N) C[row * N + col] = from_f32<TC>(moe_gated(acc[0][mt][i], acc[1][mt][i], act, rw));
                    }
                } else {
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int col = n0 + nt * 16 + 4 * g + i;
                            if (col < N) C[row * N + col] = from_f32<TC>(moe_ungated(acc[nt][mt][i], act));
                        }
                }
            }
        }
        t += run;
    }
}

// Many rows per expert, K in whole steps of 64: a block has one group of up to 8 row tiles (128 sorted rows of one expert) and 128
// rows of W (gated: the gate and up rows of 64 columns); both operands go through LDS and are shared by its four waves (2 x 2, each 64
// x 64 of the products), two LDS stages of a step of 64 of K, two steps' pieces on their way in registers, one barrier a step.  A row
// of a stage is 128 bytes, piece p of row r lies at place p ^ (r % 8), so that neither the writes nor the operands' reads meet in a bank.
// What bounds it: LDS (a wave reads 16 KB for its 32 products of 16 cycles a step, 128 bytes a cycle and compute unit with four waves,
// beside 32 KB of writes), which two blocks per compute unit keep busy in turn.  Measured, both products of 32 experts of 2 x 1536 x 2048,
// four a token: 183 + 108 us at 2011 tokens (550 and 470 TFLOP/s; 132 us with one expert's matrices in the caches) against 286 + 175
// for the kernel above, which is left for other sizes of K; 93 + 35 at 300 tokens against 184 + 85, where the matrices' way from memory
// bounds it (4.4 TB/s).
template <bool GATED, typename TC>
__global__ __launch_bounds__(256, 2) void moe_gemm_group_kernel(TC* __restrict__ C, const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                const int* __restrict__ tile_expert, const int* __restrict__ sorted_pair,
                                                                const int* __restrict__ group, int gather, int N, int K, int gy,
                                                                long long w_stride, MoeAct act) {
    __shared__ __align__(16) bf16_t stage_[2][256 * 64];       // 128 rows of A, then 128 of W
    __shared__ int src_row[128];
    // Blocks go to the dies in turn: a die takes a run of the blocks there are in (band, columns, group of the band) order, so that
    // the blocks that read the same rows of W run beside each other, and an expert's matrix comes into one L2 once (in (group,
    // columns) order half of the L2's requests missed, 955 MB a call for 403 MB of matrices: 184 us at 2011 tokens, 32 experts of
    // 2 x 1536 x 2048, four a token)
    const int total = group[0] * gy, per = (total + MOE_DIES - 1) / MOE_DIES, idx = blockIdx.x / MOE_DIES;
    const int v = (blockIdx.x % MOE_DIES) * per + idx;
    if (idx >= per || v >= total) return;
    const int band = group[2 + 2 * (v / gy)], first = band >> 3, n_band = band & 7, in_band = v - first * gy;
    const int by = in_band / n_band, gr = group[1 + 2 * (first + in_band % n_band)];
    const int t = gr >> 4, rows = (gr & 15) * MOE_TM;
    const int e = tile_expert[t];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    if (tid < 128) {
        int src = -1;
        if (tid < rows) {
            const int p = sorted_pair[t * MOE_TM + tid];
            src = p < 0 ? -1 : (gather > 0 ? p / gather : t * MOE_TM + tid);
        }
        src_row[tid] = src;
    }
    __syncthreads();
    // staging: thread t has rows t / 8 + 32 i of A and of W, 16-byte piece t % 8.  Rows that do not exist are read as row 0 or the
    // last one: what they give is not stored
    const int sr = tid >> 3, piece = tid & 7;
    const bf16_t* ap[4];
    const bf16_t* wp[4];
    const bf16_t* We = W + (size_t)e * w_stride;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = sr + 32 * i;
        ap[i] = A + (size_t)max(src_row[row], 0) * K + 8 * piece;
        const int wrow = GATED ? (row < 64 ? min(by * 64 + row, N - 1) : N + min(by * 64 + row - 64, N - 1)) : min(by * 128 + row, N - 1);
        wp[i] = We + (size_t)wrow * K + 8 * piece;
    }
    const int to = sr * 64 + ((piece ^ (sr & 7)) * 8);
    moe_f32x4_t acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = moe_f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int steps = K / 64;
    auto fetch = [&](moe_bf16x8_t (&va)[4], moe_bf16x8_t (&vw)[4], int s) {
        const int k = min(s, steps - 1) * 64;
#pragma unroll
        for (int i = 0; i < 4; ++i) vw[i] = *reinterpret_cast<const moe_bf16x8_t*>(wp[i] + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) va[i] = *reinterpret_cast<const moe_bf16x8_t*>(ap[i] + k);
    };
    auto stage = [&](const moe_bf16x8_t (&va)[4], const moe_bf16x8_t (&vw)[4], int s) {
        bf16_t* base = stage_[s & 1] + to;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<moe_bf16x8_t*>(base + 32 * i * 64) = va[i];
            *reinterpret_cast<moe_bf16x8_t*>(base + (128 + 32 * i) * 64) = vw[i];
        }
    };
    const bool busy = wm * 64 < rows;                // a wave whose rows do not exist stages only
    auto products = [&](int s) {
        if (!busy) return;
        const bf16_t* base = stage_[s & 1];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int at = ((4 * ks + g) ^ (r & 7)) * 8;
            moe_bf16x8_t fa[4], fw[4];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const int row = GATED ? (nt < 2 ? wn * 32 + nt * 16 : 64 + wn * 32 + (nt - 2) * 16) : wn * 64 + nt * 16;
                fw[nt] = *reinterpret_cast<const moe_bf16x8_t*>(base + (128 + row + r) * 64 + at);
            }
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) fa[mt] = *reinterpret_cast<const moe_bf16x8_t*>(base + (wm * 64 + mt * 16 + r) * 64 + at);
#pragma unroll
            for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                for (int nt = 0; nt < 4; ++nt) acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[nt], fa[mt], acc[nt][mt], 0, 0, 0);
        }
    };
    moe_bf16x8_t a0[4], w0[4], a1[4], w1[4];
    fetch(a0, w0, 0);
    fetch(a1, w1, 1);
    stage(a0, w0, 0);
    __syncthreads();
    int s = 0;
    for (; s + 2 < steps; s += 2) {
        fetch(a0, w0, s + 2);
        products(s);
        stage(a1, w1, s + 1);                        // (read last in step s - 1, which every wave has left)
        __syncthreads();
        fetch(a1, w1, s + 3);
        products(s + 1);
        stage(a0, w0, s + 2);
        __syncthreads();
    }
    products(s);
    if (s + 1 < steps) {
        stage(a1, w1, s + 1);
        __syncthreads();
        products(s + 1);
    }
    const bool whole = N % 4 == 0;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        const int lrow = wm * 64 + mt * 16 + r;
        if (src_row[lrow] < 0) continue;
        const size_t row = (size_t)t * MOE_TM + lrow;
        const float rw = (GATED && act.pair_w) ? act.pair_w[sorted_pair[row]] : 1.f;
#pragma unroll
        for (int nt = 0; nt < (GATED ? 2 : 4); ++nt) {
            const int col = GATED ? by * 64 + wn * 32 + nt * 16 + 4 * g : by * 128 + wn * 64 + nt * 16 + 4 * g;
            float y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = GATED ? moe_gated(acc[nt][mt][i], acc[GATED ? nt + 2 : nt][mt][i], act, rw) : moe_ungated(acc[nt][mt][i], act);
            TC* c = C + row * N + col;
            if (whole) {
                if (col < N) Vec4<TC>::store(c, y);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (col + i < N) c[i] = from_f32<TC>(y[i]);
            }
        }
    }
}

// Many rows per expert, the experts' matrices in operand order: as in gemm_rows.hip (the comments on the data flow and the waits are
// there), a block has a group's rows and 256 rows of W (gated: the gate and up rows of 128 columns), a wave all of the group's rows and 64
// of W's; W goes from memory straight into operand registers, the gathered rows of A through two LDS stages, which carry half of what the
// kernel above needs, whose bound they are.  Groups of fewer rows take fewer products: a block goes by two, four, six or eight row tiles.
// Measured, both products, us, the kernel above / this one: 32 experts of 2 x 1536 x 2048 with 16 rows each 136 / 118, 64 rows 151 / 136,
// 251 rows 268 / 235, 500 rows 470 / 371; 32 of 2 x 3072 x 4096 with 251 rows 980 / 745 (840 TFLOP/s), with 16 435 / 397 (6.1 TB/s); with
// the same rows of W loaded from row order, 64 bytes of 16 rows a load, 322 for 268 of the first ones' 251 rows.
#define MOE_HALVES 128
template <int MT, bool GATED, typename TC>
__device__ __forceinline__ void moe_rows_block(TC* C, const bf16_t* A, unsigned a_bytes, const bf16_t* We, const int* src_row, const float* row_w,
                                               bf16_t* stage0, bf16_t* stage1, int N, int K, int by, int t, const MoeAct& act) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NT = N / 16;
    const auto wres = __builtin_amdgcn_make_buffer_rsrc((void*)We, 0, (GATED ? 2 : 1) * N * K * 2, 0x00020000);
    const auto ares = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, a_bytes, 0x00020000);
    const int w_lane = lane * 16, w_turn = (GATED ? 2 : 1) * N * 256;
    int w_at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int tile = GATED ? (j >> 1) * NT + min(by * 8 + wave * 2 + (j & 1), NT - 1) : min(by * 16 + wave * 4 + j, NT - 1);
        w_at[j] = __builtin_amdgcn_readfirstlane(tile * 4096);
    }
    const int s_row = wave * 4 + (lane >> 4), s_piece = ((lane & 15) ^ s_row) * 16;
    int a_lane[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) a_lane[i] = max(src_row[i * 16 + s_row], 0) * K * 2 + s_piece;
    moe_f32x4_t acc[4][MT];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = moe_f32x4_t{0.f, 0.f, 0.f, 0.f};
    moe_bf16x8_t w[4][4];
    auto load_a = [&](bf16_t* stage, int c) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, (__attribute__((address_space(3))) void*)(stage + (i * 4 + wave) * 512), 16, a_lane[i], c * 256, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_w = [&](int s, int c) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[s][j] = __builtin_bit_cast(moe_bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(wres, w_lane, w_at[j] + c * w_turn + s * 1024, 0));
    };
    auto products = [&](const bf16_t* stage, int next, bool more) {
        const bf16_t* ab = stage + r * 128;
        moe_bf16x8_t a[4];
#pragma unroll
        for (int q = 0; q < 3; ++q) a[q] = *reinterpret_cast<const moe_bf16x8_t*>(ab + (q % MT) * 2048 + ((4 * (q / MT) + g) ^ r) * 8);
#pragma unroll
        for (int q = 0; q < 4 * MT; ++q) {
            const int s = q / MT, i = q % MT, ahead = q + 3;
            if (ahead < 4 * MT) a[ahead % 4] = *reinterpret_cast<const moe_bf16x8_t*>(ab + (ahead % MT) * 2048 + ((4 * (ahead / MT) + g) ^ r) * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][j], a[q % 4], acc[j][i], 0, 0, 0);
            if (i == MT - 1 && more) load_w(s, next);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto turn = [&]() {                               // (the 16 loads of W are a turn's last)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    const int n = K / 128;
    load_a(stage0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) load_w(s, 0);
    turn();
    int c = 0;
    for (; c + 1 < n; c += 2) {
        load_a(stage1, c + 1);
        products(stage0, c + 1, true);
        turn();
        const int after = min(c + 2, n - 1);
        load_a(stage0, after);
        products(stage1, after, true);
        turn();
    }
    if (c < n) products(stage0, 0, false);
    const int64_t row0 = (int64_t)t * MOE_TM;
    if constexpr (GATED) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (src_row[i * 16 + r] < 0) continue;
            const float rw = row_w[i * 16 + r];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int tile = by * 8 + wave * 2 + j;
                if (tile >= NT) continue;
                float y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = moe_gated(acc[j][i][e], acc[j + 2][i][e], act, rw);
                Vec4<TC>::store(C + (row0 + i * 16 + r) * N + tile * 16 + 4 * g, y);
            }
        }
    } else {
        // (nothing under way into the stages, and nobody reads them)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        // (bfloat16 results of experts without a gate, eight values of the exact gelu a turn: 28 bytes of scratch, on the way out only.  Four a turn have none and
        // take as long or 2 % longer: both products of 32 experts of 768 x 1024, 50 rows each 51.4 / 52.7 us, 1536 x 2048, 250 rows 195 / 196, 3072 x
        // 4096, 125 rows 451 / 444; formed where the sums lie, without LDS 54.5, 203 and 450.)
        constexpr int VEC = 16 / sizeof(TC);
        gr_results<MT, 8, false>(acc, stage0, C, N, N, by * 256 + wave * 64, lane, wave, [&](int, float (&v)[VEC], float (&)[VEC]) {
            if (act.kind != 2) return;
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[e] = gelu_f(v[e]);
        }, [&](int row) { return src_row[row] < 0 ? (int64_t)-1 : row0 + row; });
    }
}

template <bool GATED, typename TC>
__global__ __launch_bounds__(256, 2) void moe_gemm_rows_kernel(TC* C, const bf16_t* A, unsigned a_bytes, const bf16_t* W, const int* tile_expert,
                                                               const int* sorted_pair, const int* group, int gather, int N, int K, int gy,
                                                               long long w_stride, MoeAct act) {
    __shared__ __align__(1024) bf16_t stage0[128 * 128];
    __shared__ __align__(1024) bf16_t stage1[128 * 128];
    __shared__ int src_row[128];
    __shared__ float row_w[128];
    // (blocks to the dies in runs of the (band, columns, group of the band) order, as above)
    // Up to MOE_HALVES blocks, which leave half of the compute units idle, become two with half of their group's rows (2 experts of 2 x
    // 1536 x 2048 with 128 rows each: 38 us for both products, 64 without; 8 of 2 x 4096 x 2048: 138, 151; with a line at 256 blocks 8
    // experts with 64 rows take 122, 107 without)
    const int total = group[0] * gy, halves = total <= MOE_HALVES ? 2 : 1, per = (total + MOE_DIES - 1) / MOE_DIES, idx = blockIdx.x / MOE_DIES;
    const int half = idx >= per, v = (blockIdx.x % MOE_DIES) * per + (half ? idx - per : idx);
    if (idx >= per * halves || v >= total) return;
    const int band = group[2 + 2 * (v / gy)], first = band >> 3, n_band = band & 7, in_band = v - first * gy;
    const int by = in_band / n_band, gr = group[1 + 2 * (first + in_band % n_band)], skip = half * (MOE_GROUP / 2);
    const int t = (gr >> 4) + skip, tiles = halves == 1 ? gr & 15 : min((gr & 15) - skip, MOE_GROUP / 2);
    if (tiles <= 0) return;
    const bf16_t* We = W + (size_t)tile_expert[t] * w_stride;
    if (threadIdx.x < 128) {
        int src = -1;
        float weight = 1.f;
        if ((int)threadIdx.x < tiles * MOE_TM) {
            const int p = sorted_pair[t * MOE_TM + threadIdx.x];
            src = p < 0 ? -1 : (gather > 0 ? p / gather : t * MOE_TM + (int)threadIdx.x);
            if (GATED && act.pair_w && p >= 0) weight = act.pair_w[p];
        }
        src_row[threadIdx.x] = src;
        row_w[threadIdx.x] = weight;
    }
    __syncthreads();
    if (tiles > 6) moe_rows_block<8, GATED>(C, A, a_bytes, We, src_row, row_w, stage0, stage1, N, K, by, t, act);
    else if (tiles > 4) moe_rows_block<6, GATED>(C, A, a_bytes, We, src_row, row_w, stage0, stage1, N, K, by, t, act);
    else if (tiles > 2) moe_rows_block<4, GATED>(C, A, a_bytes, We, src_row, row_w, stage0, stage1, N, K, by, t, act);
    else moe_rows_block<2, GATED>(C, A, a_bytes, We, src_row, row_w, stage0, stage1, N, K, by, t, act);
}

static int moe_gemm_mfma_launch(void* C, int c_dtype, const void* A, const void* W, const int* tile_expert, const int* sorted_pair,
                                int gather, int gated, int tiled, bool many, int max_tiles, int N, int K, MoeAct act, hipStream_t st) {
    const long long ws = (long long)(gated ? 2 : 1) * N * K;
    if (many && !tiled) {
        const dim3 grid((max_tiles + 7) / 8, (N + (gated ? 63 : 127)) / (gated ? 64 : 128));
        SPY_REQUIRE(grid.y <= 65535, "spy_moe_gemm: too many columns");
        if (gated) {
            SPY_DISPATCH(c_dtype, TC, (moe_gemm_mfma_lds_kernel<true, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (const bf16_t*)W, tile_expert,
                                                                                               sorted_pair, gather, max_tiles, N, K, ws, act)));
        } else {
            SPY_DISPATCH(c_dtype, TC, (moe_gemm_mfma_lds_kernel<false, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (const bf16_t*)W, tile_expert,
                                                                                                sorted_pair, gather, max_tiles, N, K, ws, act)));
        }
        return 0;
    }
    const dim3 grid((N + (gated ? 15 : 31)) / (gated ? 16 : 32), max_tiles);
    SPY_REQUIRE(grid.y <= 65535, "spy_moe_gemm: too many row tiles");
#define MOE_TILE_LAUNCH(G, TILED)                                                                                                     \
    SPY_DISPATCH(c_dtype, TC, (moe_gemm_tile_kernel<G, TILED, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (const bf16_t*)W, tile_expert, \
                                                                                        sorted_pair, gather, N, K, ws, act)))
    if (gated && tiled) { MOE_TILE_LAUNCH(true, true); }
    else if (gated) { MOE_TILE_LAUNCH(true, false); }
    else if (tiled) { MOE_TILE_LAUNCH(false, true); }
    else { MOE_TILE_LAUNCH(false, false); }
#undef MOE_TILE_LAUNCH
    return 0;
}

// byte offsets within an operand are 31 bits wide in the kernel for groups of rows and matrices in operand order (beyond: a tile at a time)
static int64_t moe_a_bytes(int gather, int P, int max_tiles, int K) { return 2LL * K * (gather > 0 ? P / gather : (int64_t)max_tiles * MOE_TM); }
static bool moe_rows_fit(int gather, int P, int max_tiles, int gated, int N, int K) {
    return moe_a_bytes(gather, P, max_tiles, K) < (1LL << 31) && (int64_t)(gated ? 2 : 1) * N * K * 2 < (1LL << 31);
}

// w_tiled: every expert's matrix lies in operand order (bfloat16, whole tiles of 16 rows and whole steps of 128 of K)
extern "C" int spy_moe_gemm(void* C, int c_dtype, const void* A, int a_dtype, const void* W, int w_dtype, int w_tiled, const int* tile_expert,
                            const int* sorted_pair, const int* group, int P, int gather, int gated, int max_tiles, int E, int N, int K,
                            int tiles_per_block, int act_kind, float limit, const float* pair_w, hipStream_t st) {
    SPY_REQUIRE(max_tiles > 0 && E > 0 && N > 0 && K > 0 && gather >= 0, "spy_moe_gemm: bad sizes (%d tiles)", max_tiles);
    SPY_REQUIRE((act_kind == 0 && !pair_w) || (act_kind == 1 && gated && limit > 0.f) || (act_kind == 2 && !gated && !pair_w), "spy_moe_gemm: activation %d with limit %g", act_kind, (double)limit);
    const MoeAct act = {act_kind, limit, pair_w};
    // bfloat16 operands in 16-byte pieces: the matrix cores; tiles_per_block: 0 = the plain float32 kernel
    SPY_REQUIRE(!w_tiled || (w_dtype == SPY_BF16 && K % 128 == 0 && N % 16 == 0 && ((uintptr_t)W % 16) == 0),
                "spy_moe_gemm: matrices of %d x %d (dtype %d) do not lie in operand order", N, K, w_dtype);
    if (tiles_per_block >= 8 && group && a_dtype == SPY_BF16 && w_dtype == SPY_BF16 && K % 64 == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16) == 0 && (!w_tiled || moe_rows_fit(gather, P, max_tiles, gated, N, K))) {
        const bool wide = w_tiled != 0;
        const int cols = wide ? (gated ? 128 : 256) : (gated ? 64 : 128), gy = (N + cols - 1) / cols;
        const int64_t blocks = (int64_t)moe_max_groups(max_tiles, E, P) * gy;
        SPY_REQUIRE(blocks < (1 << 30), "spy_moe_gemm: too many blocks");
        // (up to MOE_HALVES blocks become two each, every die with its whole run twice)
        const int64_t runs = (blocks + MOE_DIES - 1) / MOE_DIES, halved = 2 * ((min(blocks, (int64_t)MOE_HALVES) + MOE_DIES - 1) / MOE_DIES);
        const unsigned grid = (unsigned)((wide ? max(runs, halved) : runs) * MOE_DIES);
        const long long ws = (long long)(gated ? 2 : 1) * N * K;
        if (wide && gated) {
            SPY_DISPATCH(c_dtype, TC, (moe_gemm_rows_kernel<true, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (unsigned)moe_a_bytes(gather, P, max_tiles, K), (const bf16_t*)W, tile_expert,
                                                                                           sorted_pair, group, gather, N, K, gy, ws, act)));
        } else if (wide) {
            SPY_DISPATCH(c_dtype, TC, (moe_gemm_rows_kernel<false, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (unsigned)moe_a_bytes(gather, P, max_tiles, K), (const bf16_t*)W, tile_expert,
                                                                                            sorted_pair, group, gather, N, K, gy, ws, act)));
        } else if (gated) {
            SPY_DISPATCH(c_dtype, TC, (moe_gemm_group_kernel<true, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (const bf16_t*)W, tile_expert, sorted_pair,
                                                                                            group, gather, N, K, gy, ws, act)));
        } else {
            SPY_DISPATCH(c_dtype, TC, (moe_gemm_group_kernel<false, TC><<<grid, 256, 0, st>>>((TC*)C, (const bf16_t*)A, (const bf16_t*)W, tile_expert, sorted_pair,
                                                                                             group, gather, N, K, gy, ws, act)));
        }
        SPY_CHECK_LAUNCH("spy_moe_gemm (groups)");
        return 0;
    }
    if (tiles_per_block > 0 && a_dtype == SPY_BF16 && w_dtype == SPY_BF16 && K % 8 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0) {
        const int rc = moe_gemm_mfma_launch(C, c_dtype, A, W, tile_expert, sorted_pair, gather, gated, w_tiled, tiles_per_block >= 8, max_tiles, N, K, act, st);
        if (rc) return rc;
        SPY_CHECK_LAUNCH("spy_moe_gemm (mfma)");
        return 0;
    }
    SPY_REQUIRE(max_tiles <= 65535, "spy_moe_gemm: %d tiles are too many for the plain kernel", max_tiles);
    const dim3 grid((N + MG_TN - 1) / MG_TN, max_tiles);
    const long long ws = (long long)(gated ? 2 : 1) * N * K;
#define MOE_PLAIN_LAUNCH(TW, G, TILED)                                                                                                   \
    SPY_DISPATCH(a_dtype, TA, SPY_DISPATCH(c_dtype, TC, (moe_gemm_kernel<TA, TW, TC, G, TILED><<<grid, 256, 0, st>>>(                     \
        (TC*)C, (const TA*)A, (const TW*)W, tile_expert, sorted_pair, gather, N, K, ws, act))))
    if (gated && w_tiled) { MOE_PLAIN_LAUNCH(bf16_t, true, true); }
    else if (w_tiled) { MOE_PLAIN_LAUNCH(bf16_t, false, true); }
    else if (gated) { SPY_DISPATCH(w_dtype, TW, MOE_PLAIN_LAUNCH(TW, true, false)); }
    else { SPY_DISPATCH(w_dtype, TW, MOE_PLAIN_LAUNCH(TW, false, false)); }
#undef MOE_PLAIN_LAUNCH
    SPY_CHECK_LAUNCH("spy_moe_gemm");
    return 0;
}

// out[t, :] = scale * sum_k weights[t, k] * Y[pair_row[t top + k], :], added in ascending k (no weights: all one); add != null:
// plus add[t, :], the result of a layer that every token uses, in the same pass
template <typename TC, bool VEC>
__global__ void moe_combine_kernel(TC* __restrict__ out, const float* __restrict__ Y, const float* __restrict__ weights,
                                   const int* __restrict__ pair_row, int top, int H, const TC* __restrict__ add, float scale) {
    // a block has one token and a run of columns (blockIdx.y): few tokens still spread over the device.  VEC: a thread has
    // four neighbouring columns (H % 4 == 0 and 16-byte aligned rows, checked by the launcher), else one.
    constexpr int N = VEC ? 4 : 1;
    const int t = blockIdx.x;
    const int c = (blockIdx.y * blockDim.x + threadIdx.x) * N;
    if (c >= H) return;
    float acc[N] = {};
    for (int k = 0; k < top; ++k) {
        const int row = pair_row[(size_t)t * top + k];
        if (row < 0) continue;
        const float w = (weights ? weights[(size_t)t * top + k] : 1.f) * scale;
        float y[N];
        if (VEC) Vec4<float>::load(Y + (size_t)row * H + c, y); else y[0] = Y[(size_t)row * H + c];
#pragma unroll
        for (int e = 0; e < N; ++e) acc[e] = fmaf(w, y[e], acc[e]);
    }
    if (add) {
        float a[N];
        if (VEC) Vec4<TC>::load(add + (size_t)t * H + c, a); else a[0] = to_f32<TC>(add[(size_t)t * H + c]);
#pragma unroll
        for (int e = 0; e < N; ++e) acc[e] += a[e];
    }
    if (VEC) Vec4<TC>::store(out + (size_t)t * H + c, acc); else out[(size_t)t * H + c] = from_f32<TC>(acc[0]);
}

extern "C" int spy_moe_combine(void* out, int dtype, const float* Y, const float* weights, const int* pair_row, int T, int top, int H,
                               const void* add, float scale, hipStream_t st) {
    SPY_REQUIRE(T > 0 && top > 0 && H > 0, "spy_moe_combine: empty operand");
    const bool vec = H % 4 == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)Y % 16) == 0 && ((uintptr_t)add % 16) == 0;
    const int per_block = vec ? 512 : 128;
    const dim3 grid(T, (H + per_block - 1) / per_block);
    SPY_REQUIRE(grid.y <= 65535, "spy_moe_combine: rows of %d values are too long", H);
    if (vec) {
        SPY_DISPATCH(dtype, TC, (moe_combine_kernel<TC, true><<<grid, 128, 0, st>>>((TC*)out, Y, weights, pair_row, top, H, (const TC*)add, scale)));
    } else {
        SPY_DISPATCH(dtype, TC, (moe_combine_kernel<TC, false><<<grid, 128, 0, st>>>((TC*)out, Y, weights, pair_row, top, H, (const TC*)add, scale)));
    }
    SPY_CHECK_LAUNCH("spy_moe_combine");
    return 0;
}
