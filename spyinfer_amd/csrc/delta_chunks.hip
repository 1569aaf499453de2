// The gated delta rule, S = diag(g) S; u = beta (v - S^T k); S = S + k u^T; o = S^T q, over chunks of 16 tokens.
//
// Token by token (matrix_memory.hip) its time is tokens times the length of one token's chain, 1.1 us.  Within a chunk that starts
// from S0, with G_t the product of the decays up to t (per key channel, from the chunk's start):
//   S_t = diag(G_t) S0 + sum_{s <= t} diag(G_t / G_s) k_s u_s^T
//   u_t = beta_t (v_t - S0^T (G_t k_t) - sum_{s < t} A_ts u_s),   A_ts = sum_c k_t[c] k_s[c] G_t[c] / G_s[c]
//   o_t = S0^T (G_t q_t) + sum_{s <= t} B_ts u_s,                 B_ts = sum_c q_t[c] k_s[c] G_t[c] / G_s[c]
// so with M = (I + diag(beta) A)^-1 diag(beta), lower triangular, u = M V - (M W) S0 with W_t = G_t k_t.  Everything but the products
// with S0 is known for all chunks at once:
//   delta_chunk_prepare   a block per (chunk, head): A, B, M and from them MV = M V, MW = M W, Q_t = G_t q_t, K_s = G_15 / G_s k_s (stored
//                         [channel][token]), G_15, into a workspace.  The quotients of decays are never formed as quotients, which
//                         underflow: they are powers of two of differences of sums of logarithms, sums in 64 bits.
//   delta_chunk_walk      a block per (entry, head, 16 value channels), a wave per 16 key channels (or 32), whose rows of S it has in
//                         registers.  Per chunk, on v_mfma_f32_16x16x4_f32: its part of MW S0 and of Q S0, the parts of u met in
//                         LDS, S = G_15 S + K^T u, and B u for the read-out, whose parts meet one chunk later.
// The result's layout (lane (column r, g): rows 4 g + i) is the second operand's layout of the next product, so S and u go from product to
// product without a move.  All of it is float32 (the sums of logarithms float64), as the token walk is.
// What bounds it: the walk's chain of about 2000 cycles a chunk (4 products, LDS, 4 products, the read-out's way through LDS), 94 times for
// 1500 tokens, not its operands' way (95 us, 92 with every chunk's from one place); the preparation's 136 x d powers of two a chunk.  Chunks
// of 16 because a chunk's tokens are then one matrix tile; the preparation grows with the square.
// Measured: 1500 tokens, 16 heads of 128 x 128: 51 us of preparation and 95 us of walk a layer (104 by four waves with 32 key channels each)
// against 1712 us token by token.  Four waves with two tiles of channels each where the delta rule's blocks outnumber the compute units: every
// wave reads all waves' parts of u out of LDS, four times as much by eight waves.  16 heads of 128 x 128, preparation and walk, four / eight: entries of 300,
// 20 and 411 tokens (384 blocks) 98 / 109, eight of 64 72 / 76, two of 300 (256 blocks) 82 / 81.5; 4 heads of 128 x 256, 32 of 40 73 / 81.5.  (The
// mLSTM, which has no such parts, is faster by eight at any number: 12 entries of 150, 8 heads of 128 x 256, 109 / 104.)
// The mLSTM, S = a S + b k v^T with numbers a and b a token, is the same with nothing taken back: u = v, B_ts = b_s G_t / G_s (q_t . k_s), K_s =
// b_s G_15 / G_s k_s, and its vector n = a n + b k goes along in the lanes' registers (a lane has the rows of n that it has of Q as an
// operand, so n . q costs eight products a lane).  8 heads of 128 x 256, 1500 tokens: a walk
// of 94 us (118 by four waves that asked for the read-out's two numbers a token where they needed them), 165 us a layer with scalars and preparation, against 765 for pieces of 64 tokens walked twice and folded.
#include "delta_chunks.h"
#include <math.h>

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float dc_f32x4_t;

#define DC_TOKENS 16
// Chunks that are prepared and walked at a time, which bounds the workspace: 128, or as many as 64 MB hold (150 chunks of 70 KB, 60
// entries of 24 tokens with 4 heads of 64 x 64: 51 us for the delta rule in two segments, 40 in one)
#define DC_SEGMENT 128
#define DC_SEGMENT_BYTES (64 << 20)

// An entry's chunks have neighbouring numbers from cu_q[e] / 16 + e on (entries' ranges cannot meet: they have at most
// cu_q[e + 1] / 16 - cu_q[e] / 16 + 1 chunks); some numbers belong to nobody.
__device__ __forceinline__ int dc_first(const int* cu_q, int e) { return cu_q[e] / DC_TOKENS + e; }
static int64_t dc_numbers(int S, int T) { return (int64_t)T / DC_TOKENS + S; }

// floats of one (chunk, head) in the workspace: MW [16][d], Q [16][d], K [d][16], MV [16][dv], B [16][16], G [d]
__device__ __host__ __forceinline__ int dc_record(int d, int dv) { return 48 * d + 16 * dv + 256 + d; }

static int64_t dc_segment(int H, int d, int dv) {
    const int64_t n = DC_SEGMENT_BYTES / ((int64_t)H * dc_record(d, dv) * 4);
    return n > DC_SEGMENT ? n : DC_SEGMENT;
}

__device__ __forceinline__ float dc_pow2(float x) { return __builtin_amdgcn_exp2f(x); }

// The entry that chunk `number` is of, by all threads of a block together; -1: nobody's
__device__ __forceinline__ int dc_entry(const int* cu_q, int S, int number, int* shared) {
    if (threadIdx.x == 0) *shared = -1;
    __syncthreads();
    for (int e = threadIdx.x; e < S; e += 256) {
        const int f = dc_first(cu_q, e), n = cu_q[e + 1] - cu_q[e];
        if (number >= f && number < f + (n + DC_TOKENS - 1) / DC_TOKENS) *shared = e;
    }
    __syncthreads();
    return *shared;
}

template <typename TA, int D>
__global__ __launch_bounds__(256) void delta_chunk_prepare_kernel(DeltaChunks a, int number0) {
    __shared__ __align__(16) float kk[16][D + 4], qq[16][D + 4];
    __shared__ __align__(16) double ll[16][D + 2];
    __shared__ __align__(16) float A[16][20], M[16][20];
    __shared__ float beta[16];
    __shared__ int shared;
    const int number = number0 + blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int entry = dc_entry(a.cu_q, a.S, number, &shared);
    if (entry < 0) return;
    const int t0 = a.cu_q[entry] + (number - dc_first(a.cu_q, entry)) * DC_TOKENS, n = min(DC_TOKENS, a.cu_q[entry + 1] - t0);
    const int g = h / (a.H / a.G);
    // tokens beyond the entry's end: k, q, v and beta zero, no decay
    for (int i = tid; i < 16 * D; i += 256) {
        const int t = i / D, c = i % D;
        const float* row = a.qk + (size_t)(t0 + t) * 2 * a.G * D + c;
        qq[t][c] = t < n ? row[(size_t)g * D] : 0.f;
        kk[t][c] = t < n ? row[(size_t)(a.G + g) * D] : 0.f;
        const float z = t < n ? a.dec[(size_t)(t0 + t) * a.zs + (size_t)h * a.dd + (a.dd == 1 ? 0 : c)] : 1.f;
        const float l = log2f(z);
        ll[t][c] = (double)(l < -1e5f ? -1e5f : l);         // (a decay of zero is 2^-100000: zero in every product, and differences stay numbers)
    }
    if (tid < 16) beta[tid] = tid < n ? a.beta[(size_t)(t0 + tid) * a.bs + h] : 0.f;
    __syncthreads();
    if (tid < D) {
        double sum = 0.0;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            sum += ll[t][tid];
            ll[t][tid] = sum;
        }
    }
    __syncthreads();
    float* out = a.ws + ((size_t)blockIdx.x * a.H + h) * dc_record(D, a.dv);
    float* o_mw = out;
    float* o_q = o_mw + 16 * D;
    float* o_k = o_q + 16 * D;
    float* o_mv = o_k + 16 * D;
    float* o_b = o_mv + 16 * a.dv;
    float* o_g = o_b + 256;
    {   // thread (t, s): A and B of the pair
        const int t = tid >> 4, s = tid & 15;
        float x = 0.f, y = 0.f;
        if (s <= t) {
            for (int c = 0; c < D; c += 4) {
                const dc_f32x4_t kt = *reinterpret_cast<const dc_f32x4_t*>(&kk[t][c]), ks = *reinterpret_cast<const dc_f32x4_t*>(&kk[s][c]);
                const dc_f32x4_t qt = *reinterpret_cast<const dc_f32x4_t*>(&qq[t][c]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float w = ks[e] * dc_pow2((float)(ll[t][c + e] - ll[s][c + e]));
                    x = fmaf(kt[e], w, x);
                    y = fmaf(qt[e], w, y);
                }
            }
        }
        A[t][s] = s < t ? x : 0.f;
        o_b[t * 16 + s] = y;                                // (zero above the diagonal)
    }
    __syncthreads();
    if (tid < 16) {                                         // column tid of M, forwards
        float m[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float x = t == tid ? 1.f : 0.f;
#pragma unroll
            for (int s = 0; s < t; ++s) x = fmaf(-A[t][s], m[s], x);
            m[t] = beta[t] * x;
            M[t][tid] = m[t];
        }
    }
    __syncthreads();
    // a thread per column of W or V: the column of M W or M V
    for (int i = tid; i < D + a.dv; i += 256) {
        float x[16];
        if (i < D) {
#pragma unroll
            for (int s = 0; s < 16; ++s) x[s] = kk[s][i] * dc_pow2((float)ll[s][i]);
        } else {
            const TA* v = (const TA*)a.qkv + (size_t)t0 * (2 * a.G * D + a.H * a.dv) + 2 * a.G * D + (size_t)h * a.dv + (i - D);
#pragma unroll
            for (int s = 0; s < 16; ++s) x[s] = s < n ? to_f32<TA>(v[(size_t)s * (2 * a.G * D + a.H * a.dv)]) : 0.f;
        }
        float* to = i < D ? o_mw + i : o_mv + (i - D);
        const int ld = i < D ? D : a.dv;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float y = 0.f;
#pragma unroll
            for (int s = 0; s <= t; ++s) y = fmaf(M[t][s], x[s], y);
            to[(size_t)t * ld] = y;
        }
    }
    for (int i = tid; i < 16 * D; i += 256) {
        o_q[i] = qq[i / D][i % D] * dc_pow2((float)ll[i / D][i % D]);
        const int c = i / 16, s = i % 16;
        o_k[i] = kk[s][c] * dc_pow2((float)(ll[15][c] - ll[s][c]));
    }
    if (tid < D) o_g[tid] = dc_pow2((float)ll[15][tid]);
}

// The mLSTM's chunks: the same records, with the sum of K over the chunk's tokens [d], the sums of B's rows [16] and e^-m [16] in MW's place.
template <typename TA, int D>
__global__ __launch_bounds__(256) void memory_chunk_prepare_kernel(MemoryChunks a, int number0) {
    __shared__ __align__(16) float kk[16][D + 4], qq[16][D + 4];
    __shared__ __align__(16) float B[16][20];
    __shared__ double ll[16];
    __shared__ float b[16];
    __shared__ int shared;
    const int number = number0 + blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int entry = dc_entry(a.cu_q, a.S, number, &shared);
    if (entry < 0) return;
    const int t0 = a.cu_q[entry] + (number - dc_first(a.cu_q, entry)) * DC_TOKENS, n = min(DC_TOKENS, a.cu_q[entry + 1] - t0);
    const float qscale = 1.0f / sqrtf((float)D);
    for (int i = tid; i < 16 * D; i += 256) {
        const int t = i / D, c = i % D;
        const TA* row = (const TA*)a.x + (size_t)(t0 + t) * a.xs + (size_t)h * D + c;
        qq[t][c] = t < n ? to_f32<TA>(row[a.q_off]) * qscale : 0.f;
        kk[t][c] = t < n ? to_f32<TA>(row[a.k_off]) : 0.f;
    }
    float* out = a.ws + ((size_t)blockIdx.x * a.H + h) * dc_record(D, a.dv);
    float* o_q = out + 16 * D;
    float* o_k = o_q + 16 * D;
    float* o_v = o_k + 16 * D;
    float* o_b = o_v + 16 * a.dv;
    float* o_g = o_b + 256;
    if (tid < 16) {
        const float* g = a.abe + (size_t)(t0 + tid) * 3 * a.H + h;
        const float l = tid < n ? log2f(g[0]) : 0.f;
        double sum = (double)(l < -1e5f ? -1e5f : l);
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const double x = __shfl_up(sum, o, 16);
            if (tid >= o) sum += x;
        }
        ll[tid] = sum;
        b[tid] = tid < n ? g[a.H] : 0.f;
        out[D + 16 + tid] = tid < n ? g[2 * a.H] : 1.f;
    }
    __syncthreads();
    {
        const int t = tid >> 4, s = tid & 15;
        float y = 0.f, y2 = 0.f;
        if (s <= t) {
            for (int c = 0; c < D; c += 4) {
                const dc_f32x4_t qt = *reinterpret_cast<const dc_f32x4_t*>(&qq[t][c]), ks = *reinterpret_cast<const dc_f32x4_t*>(&kk[s][c]);
                y = fmaf(qt[0], ks[0], y); y2 = fmaf(qt[1], ks[1], y2);
                y = fmaf(qt[2], ks[2], y); y2 = fmaf(qt[3], ks[3], y2);
            }
            y = (y + y2) * (b[s] * dc_pow2((float)(ll[t] - ll[s])));
        }
        o_b[t * 16 + s] = y;
        B[t][s] = y;
    }
    for (int i = tid; i < 16 * D; i += 256) {
        o_q[i] = qq[i / D][i % D] * dc_pow2((float)ll[i / D]);
        const int c = i / 16, s = i % 16;
        o_k[i] = kk[s][c] * (b[s] * dc_pow2((float)(ll[15] - ll[s])));
    }
    for (int i = tid; i < 16 * a.dv; i += 256) {
        const int t = i / a.dv, c = i % a.dv;
        o_v[i] = t < n ? to_f32<TA>(((const TA*)a.x)[(size_t)(t0 + t) * a.xs + a.v_off + (size_t)h * a.dv + c]) : 0.f;
    }
    if (tid < D) {
        o_g[tid] = dc_pow2((float)ll[15]);
        float sum = 0.f;
#pragma unroll
        for (int s = 0; s < 16; ++s) sum = fmaf(kk[s][tid], b[s] * dc_pow2((float)(ll[15] - ll[s])), sum);
        out[tid] = sum;
    }
    __syncthreads();
    if (tid < 16) {
        float sum = 0.f;
        for (int s = 0; s <= tid; ++s) sum += B[tid][s];
        out[D + tid] = sum;
    }
}

// What the walk needs of either recurrence
struct ChunkWalk {
    float* o;
    float* state;
    long long slot_stride, head_stride;
    const float* mfin;
    const int* cu_q;
    const int* slot_ids;
    int num_slots, H, dv;
    const float* ws;
};

template <int D, bool DELTA, int TI>
__global__ __launch_bounds__(D * 4 / TI) void chunk_walk_kernel(ChunkWalk a, int number0, int number1) {
    constexpr int W = D / (16 * TI);                        // waves, each with TI tiles of 16 key channels
    constexpr int READ = W > 4 ? 4 : 0;                     // four waves multiply B by u (from 0 on), four read out (from here on)
    __shared__ __align__(16) float pu[DELTA ? 2 : 1][W][64][4], po[2][W][64][4];
    __shared__ float pn[2][W][16];
    const int e = blockIdx.x, h = blockIdx.y, col0 = blockIdx.z * 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int slot = a.slot_ids[e];
    if (slot < 0 || slot >= a.num_slots) return;
    const int q0 = a.cu_q[e], q1 = a.cu_q[e + 1], first = dc_first(a.cu_q, e), chunks = (q1 - q0 + DC_TOKENS - 1) / DC_TOKENS;
    const int c0 = max(0, number0 - first), c1 = min(chunks, number1 - first);
    if (c0 >= c1) return;
    const int row0 = wave * 16 * TI + 4 * g;                // lane (column r, g) has rows row0 + 16 i .. + 3
    float* head = a.state + (size_t)slot * a.slot_stride + (size_t)h * a.head_stride;
    float* st = head + col0 + r;
    float* nm = head + (size_t)D * a.dv + (size_t)blockIdx.z * (D + 1);          // (mLSTM)
    dc_f32x4_t S[TI], N[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            S[i][x] = st[(size_t)(row0 + 16 * i + x) * a.dv];
            N[i][x] = DELTA ? 0.f : nm[row0 + 16 * i + x];
        }
    const int rec = dc_record(D, a.dv);
    auto record = [&](int c) { return a.ws + ((size_t)(first + min(c, c1 - 1) - number0) * a.H + h) * rec; };
    // this lane's operands of a chunk (mw: the mLSTM's sums of K; nb, em: its row's sum of B and e^-m).  Their places in a record are
    // 32-bit numbers that are worked out once, beside an address that the whole block has in common.
    const int o_row = 4 * g + (wave & 3);                   // the row that the lane reads out
    const unsigned at_mw = 4u * ((DELTA ? r * D : 0) + row0), at_q = 4u * (16 * D + r * D + row0), at_k = 4u * (32 * D + (wave * 16 * TI + r) * 16 + 4 * g);
    const unsigned at_b = 4u * (48 * D + 16 * a.dv + r * 16 + 4 * g), at_g = 4u * (48 * D + 16 * a.dv + 256 + row0), at_n = 4u * (D + o_row);
    unsigned at_v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) at_v[i] = 4u * (48 * D + (4 * g + i) * a.dv + col0 + r);
    struct Ops { dc_f32x4_t mw[TI], q[TI], k[TI], gl[TI], b, mv; float nb, em; };
    auto load = [&](Ops& x, int c) {
        const char* p = reinterpret_cast<const char*>(record(c));
#pragma unroll
        for (int i = 0; i < TI; ++i) {                      // (a tile's numbers lie 16 of a row, or 16 rows of 16, behind the one before)
            x.mw[i] = *reinterpret_cast<const dc_f32x4_t*>(p + at_mw + 64 * i);
            x.q[i] = *reinterpret_cast<const dc_f32x4_t*>(p + at_q + 64 * i);
            x.k[i] = *reinterpret_cast<const dc_f32x4_t*>(p + at_k + 1024 * i);
            x.gl[i] = *reinterpret_cast<const dc_f32x4_t*>(p + at_g + 64 * i);
        }
        x.b = *reinterpret_cast<const dc_f32x4_t*>(p + at_b);
#pragma unroll
        for (int i = 0; i < 4; ++i) x.mv[i] = *reinterpret_cast<const float*>(p + at_v[i]);
        x.nb = DELTA ? 0.f : *reinterpret_cast<const float*>(p + at_n);
        x.em = DELTA ? 0.f : *reinterpret_cast<const float*>(p + at_n + 64);
    };
    // read-out of chunk c: the waves' parts, row o_row of column r
    float* const o_at = a.o + (size_t)h * a.dv + col0 + r;
    auto read_out = [&](int c, float nb, float em) {
        const int t = q0 + c * DC_TOKENS + o_row;
        float y = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) y += po[c & 1][w][lane][wave & 3];
        if (!DELTA) {
            float nq = nb;
#pragma unroll
            for (int w = 0; w < W; ++w) nq += pn[c & 1][w][o_row];
            y /= fmaxf(fabsf(nq), em) + 1e-6f;
        }
        if (t < q1) o_at[(size_t)t * a.H * a.dv] = y;
    };
    float nb = 0.f, em = 0.f;                               // of the chunk before
    auto chunk = [&](const Ops& x, int c) {
        dc_f32x4_t o0 = {0.f, 0.f, 0.f, 0.f}, o1 = {0.f, 0.f, 0.f, 0.f};
        if (DELTA) {
            dc_f32x4_t u0 = {0.f, 0.f, 0.f, 0.f}, u1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < 4; j += 2) {
                    u0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.mw[i][j], S[i][j], u0, 0, 0, 0);
                    u1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.mw[i][j + 1], S[i][j + 1], u1, 0, 0, 0);
                }
            *reinterpret_cast<dc_f32x4_t*>(pu[DELTA ? c & 1 : 0][wave][lane]) = u0 + u1;
        }
        float nq = 0.f;
        if (!DELTA) {
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) nq = fmaf(x.q[i][j], N[i][j], nq);        // lane (token r, g): its rows' share of n . q
            nq += __shfl_xor(nq, 16, 64);
            nq += __shfl_xor(nq, 32, 64);
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) N[i][j] = fmaf(x.gl[i][j], N[i][j], x.mw[i][j]);
        }
        __syncthreads();                                    // parts of u of this chunk, and of the read-out of the chunk before
        dc_f32x4_t parts[DELTA ? W : 1];
        if (DELTA) {
#pragma unroll
            for (int w = 0; w < W; ++w) parts[w] = *reinterpret_cast<const dc_f32x4_t*>(pu[DELTA ? c & 1 : 0][w][lane]);
        }
        // (Q S0 runs while the parts of u come out of LDS)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[i][j], S[i][j], o0, 0, 0, 0);
                o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[i][j + 1], S[i][j + 1], o1, 0, 0, 0);
            }
        dc_f32x4_t u = x.mv;
        if (DELTA) {
#pragma unroll
            for (int w = 0; w < W; ++w) u -= parts[w];
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) S[i] *= x.gl[i];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < TI; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][j], u[j], S[i], 0, 0, 0);
        if (wave < 4) {
            // of B u, this wave's share: tokens s = 4 g + wave
            float bw = x.b[0], uw = u[0];
#pragma unroll
            for (int j = 1; j < 4; ++j)
                if (wave == j) { bw = x.b[j]; uw = u[j]; }
            // (B is zero where a token does not read: infinities and NaN, which zero does not take away, go to the rows that do read them)
            const bool odd = !(fabsf(uw) < INFINITY);
            if (__any(odd)) {
                const dc_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
                const dc_f32x4_t f = __builtin_amdgcn_mfma_f32_16x16x4f32(4 * g + wave <= r ? 1.f : 0.f, odd ? 1.f : 0.f, zero, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (f[i] > 0.f) o0[i] = __builtin_nanf("");
                if (odd) uw = 0.f;
            }
            o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(bw, uw, o0, 0, 0, 0);
        }
        if (wave >= READ && c > c0) read_out(c - 1, nb, em);
        nb = x.nb;
        em = x.em;
        // (the place was read for chunk c - 2 behind the barrier of chunk c - 1, which every wave has passed)
        *reinterpret_cast<dc_f32x4_t*>(po[c & 1][wave][lane]) = o0 + o1;
        if (!DELTA && g == 0) pn[c & 1][wave][r] = nq;
    };
    Ops x0, x1;                                             // (three chunks' operands under way instead of one: 97 to 105 us)
    load(x0, c0);
    int c = c0;
    for (; c + 2 <= c1; c += 2) {
        load(x1, c + 1);
        chunk(x0, c);
        load(x0, c + 2);
        chunk(x1, c + 1);
    }
    if (c < c1) chunk(x0, c);
    __syncthreads();
    if (wave >= READ) read_out(c1 - 1, nb, em);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            st[(size_t)(row0 + 16 * i + y) * a.dv] = S[i][y];
            if (!DELTA && r == 0) nm[row0 + 16 * i + y] = N[i][y];
        }
    if (!DELTA && threadIdx.x == 0) nm[D] = a.mfin[(size_t)e * a.H + h];
}

bool delta_chunks_takes(int S, int T, int d, int dv) { return T > S && (d == 64 || d == 128) && dv % 16 == 0; }

int64_t delta_chunks_workspace(int S, int T, int H, int d, int dv) {
    const int64_t n = dc_numbers(S, T), most = dc_segment(H, d, dv);
    return (n < most ? n : most) * H * dc_record(d, dv);
}

int delta_chunks(const DeltaChunks& a, int dtype, hipStream_t st) {
    SPY_REQUIRE(a.ws && a.ws_floats >= delta_chunks_workspace(a.S, a.T, a.H, a.d, a.dv), "delta rule: the chunks' workspace is too small");
    SPY_REQUIRE(((uintptr_t)a.ws % 16) == 0 && a.H <= 65535 && a.dv / 16 <= 65535, "delta rule: workspace alignment or heads");
    const ChunkWalk w = {a.o, a.state, a.state_stride, (long long)a.d * a.dv, nullptr, a.cu_q, a.slot_ids, a.num_slots, a.H, a.dv, a.ws};
    const int64_t numbers = dc_numbers(a.S, a.T), segment = dc_segment(a.H, a.d, a.dv);
    for (int64_t n0 = 0; n0 < numbers; n0 += segment) {
        const int n1 = (int)(n0 + segment < numbers ? n0 + segment : numbers);
        const dim3 pgrid((unsigned)(n1 - n0), a.H), wgrid(a.S, a.H, a.dv / 16);
        if (a.d == 64) {
            SPY_DISPATCH(dtype, TA, (delta_chunk_prepare_kernel<TA, 64><<<pgrid, 256, 0, st>>>(a, (int)n0)));
            chunk_walk_kernel<64, true, 1><<<wgrid, 256, 0, st>>>(w, (int)n0, n1);
        } else {
            SPY_DISPATCH(dtype, TA, (delta_chunk_prepare_kernel<TA, 128><<<pgrid, 256, 0, st>>>(a, (int)n0)));
            // (more blocks than compute units: fewer waves, see the top)
            if ((int64_t)a.S * a.H * (a.dv / 16) > 256) chunk_walk_kernel<128, true, 2><<<wgrid, 256, 0, st>>>(w, (int)n0, n1);
            else chunk_walk_kernel<128, true, 1><<<wgrid, 512, 0, st>>>(w, (int)n0, n1);
        }
        SPY_CHECK_LAUNCH("spy_delta_rule (chunks)");
    }
    return 0;
}

int memory_chunks(const MemoryChunks& a, int dtype, hipStream_t st) {
    SPY_REQUIRE(a.ws && a.ws_floats >= delta_chunks_workspace(a.S, a.T, a.H, a.d, a.dv), "mLSTM: the chunks' workspace is too small");
    SPY_REQUIRE(((uintptr_t)a.ws % 16) == 0 && a.H <= 65535 && a.dv / 16 <= 65535, "mLSTM: workspace alignment or heads");
    const long long head = (long long)a.d * a.dv + (long long)(a.dv / 16) * (a.d + 1);
    const ChunkWalk w = {a.o, a.state, head * a.H, head, a.mfin, a.cu_q, a.slot_ids, a.num_slots, a.H, a.dv, a.ws};
    const int64_t numbers = dc_numbers(a.S, a.T), segment = dc_segment(a.H, a.d, a.dv);
    for (int64_t n0 = 0; n0 < numbers; n0 += segment) {
        const int n1 = (int)(n0 + segment < numbers ? n0 + segment : numbers);
        const dim3 pgrid((unsigned)(n1 - n0), a.H), wgrid(a.S, a.H, a.dv / 16);
        if (a.d == 64) {
            SPY_DISPATCH(dtype, TA, (memory_chunk_prepare_kernel<TA, 64><<<pgrid, 256, 0, st>>>(a, (int)n0)));
            chunk_walk_kernel<64, false, 1><<<wgrid, 256, 0, st>>>(w, (int)n0, n1);
        } else {
            SPY_DISPATCH(dtype, TA, (memory_chunk_prepare_kernel<TA, 128><<<pgrid, 256, 0, st>>>(a, (int)n0)));
            chunk_walk_kernel<128, false, 1><<<wgrid, 512, 0, st>>>(w, (int)n0, n1);
        }
        SPY_CHECK_LAUNCH("spy_mlstm (chunks)");
    }
    return 0;
}
