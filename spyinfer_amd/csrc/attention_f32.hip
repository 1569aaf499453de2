// Paged attention in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: products and sums of 32-bit numbers), for head sizes 64
// and 128 and pages of a multiple of 16 keys.  Everything that attention_generic.hip takes beside (window, chunk, cap, distance
// penalty, sink, gate), single tokens and portions alike; that kernel stands for the other shapes.
//
// A block of AF waves has a 16-row tile of one entry ((token, query head of the kv head's group) pairs, token major), one kv head
// and one part of the keys; its waves take the part's blocks of 16 keys in turn and meet through LDS.  With several parts a second
// kernel adds them.  Per block of 16 keys, lane (r = lane % 16, g = lane / 16):
//   S^T = K . Q^T     lane (key r, g) loads the values 16 s + 4 g .. of its key, lane (row r, g) holds the same of its query: product
//                     j of four takes the j-th of them.  Lane (row r, g) ends up with the scores of keys 4 g .. 4 g + 3.
//   softmax           running maximum and sum per row; only the maximum is combined over a row's four lanes
//   O^T += V^T . P^T  lane (dim r, g) loads the values of keys 4 g .. of its dim (values lie [d][key] in a page): product j takes the
//                     j-th of them and the j-th of its own four weights, so nothing moves between lanes.
//
// RAW: steps of single tokens take the step's product [q | k | v] as it is (no kernel of its own for norms, rotation and store: a step of 4 requests, 28 layers of
// 8 kv heads of 128, 1952 / 1884 us): a lane has
// of its query row the values 16 i + 4 g .., the rotation's pairs i and i + D / 32 side by side, so the norm costs two lane exchanges and the
// rotation none.  The entry's new key and value are prepared by the last wave of its last part while that wave's first keys are on their
// way: the key's score is where the wave's maximum starts, the value its result so far; the wave stores both.  Nobody reads that place.
//
// What bounds it: decoding, the round trips of one block after another (pages are looked up two blocks ahead, the next block's keys
// asked for ahead of this one's softmax, its values ahead of its scores); prompts, L2, from which a tile of 16 rows reads 1 KB a
// key of 128 dims: 8 kv heads are dealt to the 8 dies, a die's blocks reading one head's keys.
#include "common.h"
#include "attention_merge.h"
#include <math.h>

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float af_f32x4_t;
#define AF 4

struct AfArgs {
    float* out;
    const float* q;
    const float* kc;
    const float* vc;
    int P, num_pages;
    const int* cu_q;
    const int* pos0;
    const int* kv_len;
    const int* block_table;
    int max_blocks;
    const int* tile_entry;
    const int* tile_row0;
    int n_q, n_kv;
    float scale;
    int window;
    float softcap;
    int splits;
    float* ws;
    const float* dist;
    const float* sink;
    int chunk;
    const float* gate;
    long long gate_ld;
};

// The step's raw product, rows [q | k | v]; null: q comes normed and rotated.  qw, kw: the heads' norm weights (null: no norm); cos_t, sin_t: [max_pos][d / 2]
// (null: no rotation); store: this call's keys and values go to the cache (else they are there).
struct AfRaw {
    const float* qkv;
    const float* qw;
    const float* kw;
    float eps;
    const float* cos_t;
    const float* sin_t;
    int max_pos, store;
};

// One row's norm and rotation, of which lane (row, g) has the values 16 i + 4 g .. + 3
template <int DT>
__device__ __forceinline__ void af_prepare(af_f32x4_t (&x)[DT], bool normed, const af_f32x4_t (&w)[DT], float eps, bool rotated, const af_f32x4_t (&cs)[DT / 2],
                                           const af_f32x4_t (&sn)[DT / 2]) {
    if (normed) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = fmaf(x[i][e], x[i][e], ss);
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        const float scale = 1.0f / sqrtf(ss / (float)(16 * DT) + eps);
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[i][e] = (scale * x[i][e]) * w[i][e];
    }
    if (rotated) {
#pragma unroll
        for (int i = 0; i < DT / 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = x[i][e], b = x[i + DT / 2][e];
                x[i][e] = a * cs[i][e] - b * sn[i][e];
                x[i + DT / 2][e] = a * sn[i][e] + b * cs[i][e];
            }
    }
}

// the result of one row's four neighbouring dims, gated and stored
__device__ __forceinline__ void af_store(const AfArgs& a, int t, int col, int width, af_f32x4_t o, float l) {
    float4 y;
    float* v = reinterpret_cast<float*>(&y);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = l > 0.f ? o[e] / l : 0.f;
        if (a.gate) v[e] /= 1.0f + expf(-a.gate[(size_t)t * a.gate_ld + col + e]);
    }
    *reinterpret_cast<float4*>(a.out + (size_t)t * width + col) = y;
}

// (two blocks a compute unit: left to itself the compiler takes 260 registers for heads of 128 and leaves room for one)
template <int D, bool RAW>
__global__ __launch_bounds__(AF * 64, 2) void attention_f32_kernel(AfArgs a, int tiles, AfRaw z) {
    constexpr int DT = D / 16;
    __shared__ float lo_[AF][DT][64][4];
    __shared__ float lm_[AF][16], ll_[AF][16];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int hk = blockIdx.x, tile = tiles - 1 - (int)blockIdx.y, sp = blockIdx.z;      // an entry's last tile, which reads most keys, first
    // (RAW: every entry is one token and has one tile, which the caller has checked: tile t is entry t with token t)
    const int s = RAW ? tile : a.tile_entry[tile], row0 = RAW ? 0 : a.tile_row0[tile];
    const int G = a.n_q / a.n_kv;
    const int q0 = RAW ? s : a.cu_q[s], nrows = (RAW ? 1 : a.cu_q[s + 1] - q0) * G, p0 = a.pos0[s];
    const int kvl = RAW && z.store ? min(a.kv_len[s], p0) : a.kv_len[s];                  // (the new key, at p0, is not read from the cache)
    const int* bt = a.block_table + (size_t)s * a.max_blocks;
    const int row = row0 + r;
    const bool row_ok = row < nrows;
    const int tq = row_ok ? row / G : 0, head = hk * G + (row_ok ? row % G : 0);
    const int pos = row_ok ? min(p0 + tq, kvl - 1) : -1;                                  // last key of this row; none beyond the rows
    const int first = row_ok ? attention_first_key(p0 + tq, a.window, a.chunk) : 0;
    af_f32x4_t q[DT];
    {
        const float* qp = (RAW ? z.qkv + ((size_t)(q0 + tq) * (a.n_q + 2 * a.n_kv) + head) * D : a.q + ((size_t)(q0 + tq) * a.n_q + head) * D) + 4 * g;
#pragma unroll
        for (int i = 0; i < DT; ++i) q[i] = *reinterpret_cast<const af_f32x4_t*>(qp + 16 * i);
    }
    const int last_row = min(nrows, row0 + 16) - 1;
    const int hi = min(p0 + last_row / G, kvl - 1);
    const int lo = attention_first_key(p0 + row0 / G, a.window, a.chunk) & ~15;
    const int nblk = hi >= lo ? (hi - lo) / 16 + 1 : 0;
    const int per = (nblk + a.splits - 1) / a.splits;
    const int b_end = min(nblk, (sp + 1) * per);
    af_f32x4_t acc[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) acc[i] = af_f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    if (a.sink && sp == 0 && wave == 0 && row_ok) { m = a.sink[head]; l = g == 0 ? 1.f : 0.f; }
    const float d1 = a.dist ? a.dist[head] : 0.f, d2 = a.dist ? a.dist[a.n_q + head] : 0.f;
    // RAW: what the preparation needs is asked for ahead of the keys, which need the pages first
    const bool has_new = RAW && z.store && wave == AF - 1 && sp == a.splits - 1;
    constexpr int RT = RAW ? DT : 2;
    af_f32x4_t knew[RT], wq[RT], wk[RT], cs[RT / 2], sn[RT / 2];
    float vnew[RAW ? D / 64 : 1];                           // the new value's dims lane, lane + 64, for the cache
    int new_page = -1;
    if constexpr (RAW) {
        if (has_new) {
            const float* kp = z.qkv + ((size_t)q0 * (a.n_q + 2 * a.n_kv) + a.n_q + hk) * D;
            const float* vp = kp + (size_t)a.n_kv * D;
            new_page = bt[p0 / a.P];
#pragma unroll
            for (int i = 0; i < DT; ++i) {
                knew[i] = *reinterpret_cast<const af_f32x4_t*>(kp + 16 * i + 4 * g);
                acc[i] = *reinterpret_cast<const af_f32x4_t*>(vp + 16 * i + 4 * g);
                if (z.kw) wk[i] = *reinterpret_cast<const af_f32x4_t*>(z.kw + 16 * i + 4 * g);
            }
#pragma unroll
            for (int i = 0; i < D / 64; ++i) vnew[i] = vp[64 * i + lane];
        }
        if (z.qw) {
#pragma unroll
            for (int i = 0; i < DT; ++i) wq[i] = *reinterpret_cast<const af_f32x4_t*>(z.qw + 16 * i + 4 * g);
        }
        if (z.cos_t) {
            const size_t at = (size_t)max(0, min(p0, z.max_pos - 1)) * (D / 2) + 4 * g;
#pragma unroll
            for (int i = 0; i < DT / 2; ++i) {
                cs[i] = *reinterpret_cast<const af_f32x4_t*>(z.cos_t + at + 16 * i);
                sn[i] = *reinterpret_cast<const af_f32x4_t*>(z.sin_t + at + 16 * i);
            }
        }
    }

    // the page of block b of 16 keys (a page holds whole blocks); beyond the part's end the last block's
    auto page_of = [&](int b) { return bt[(lo + 16 * min(b, b_end - 1)) / a.P]; };
    auto place = [&](int b, int page, const float* base, int per_key, int lane_off) {
        const int c0 = lo + 16 * min(b, b_end - 1);
        const int pg = (page >= 0 && page < a.num_pages) ? page : 0;                       // a page that is gone: masked by position, values zeroed
        return base + (((size_t)pg * a.n_kv + hk) * a.P * D + (size_t)(c0 % a.P) * per_key) + lane_off;
    };
    int b = sp * per + wave;
    af_f32x4_t k[DT], v[DT];
    int page = 0, page_n = 0;
    {
        auto load_k = [&](int bb, int pg) {
            const float* kp = place(bb, pg, a.kc, D, r * D + 4 * g);
#pragma unroll
            for (int i = 0; i < DT; ++i) k[i] = *reinterpret_cast<const af_f32x4_t*>(kp + 16 * i);
        };
        if (b < b_end) {
            page = page_of(b);
            page_n = page_of(b + AF);
            load_k(b, page);
        }
        if constexpr (RAW) {
            af_prepare<DT>(q, z.qw != nullptr, wq, z.eps, z.cos_t != nullptr, cs, sn);
            if (has_new) {
                af_prepare<DT>(knew, z.kw != nullptr, wk, z.eps, z.cos_t != nullptr, cs, sn);
                float x = 0.f;
#pragma unroll
                for (int i = 0; i < DT; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) x = fmaf(q[i][e], knew[i][e], x);
                x += __shfl_xor(x, 16, 64);
                x += __shfl_xor(x, 32, 64);
                m = x * a.scale;
                l = g == 0 ? 1.f : 0.f;                    // (the four lanes of a row hold partial sums)
                if (new_page >= 0 && new_page < a.num_pages) {
                    const int off = p0 % a.P;
                    if (r == 0) {
                        float* to = const_cast<float*>(a.kc) + (((size_t)new_page * a.n_kv + hk) * a.P + off) * D + 4 * g;
#pragma unroll
                        for (int i = 0; i < DT; ++i) *reinterpret_cast<af_f32x4_t*>(to + 16 * i) = knew[i];
                    }
#pragma unroll
                    for (int i = 0; i < D / 64; ++i) const_cast<float*>(a.vc)[(((size_t)new_page * a.n_kv + hk) * D + 64 * i + lane) * a.P + off] = vnew[i];
                }
            }
        }
        for (; b < b_end; b += AF) {
            const int c0 = lo + 16 * b + 4 * g;                                            // this lane's four keys
            const float* vp = place(b, page, a.vc, 1, r * a.P + 4 * g);
#pragma unroll
            for (int i = 0; i < DT; ++i) v[i] = *reinterpret_cast<const af_f32x4_t*>(vp + (size_t)i * 16 * a.P);
            af_f32x4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < DT; i += 2)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][j], q[i][j], s0, 0, 0, 0);
                    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i + 1][j], q[i + 1][j], s1, 0, 0, 0);
                }
            const bool page_ok = page >= 0 && page < a.num_pages;
            page = page_n;
            page_n = page_of(b + 2 * AF);
            load_k(b + AF, page);                                                          // (behind the part's last block: that block again)
            const int n_ok = page_ok ? hi - c0 + 1 : 0;                                    // of this lane's keys, those that exist
            float sc[4], bm = -INFINITY;
            bool hidden = false;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float x = (s0[j] + s1[j]) * a.scale;
                if (a.softcap > 0.f) x = a.softcap * tanhf(x / a.softcap);
                if (a.dist) x -= d1 * log1pf(d2 * (float)(p0 + tq - (c0 + j)));
                const bool seen = c0 + j <= pos && c0 + j >= first && page_ok;
                hidden |= row_ok && !seen && j < n_ok;
                sc[j] = seen ? x : -INFINITY;
                bm = fmaxf(bm, sc[j]);
            }
            bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
            bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
            if (__any(bm > m)) {
                const float m_new = fmaxf(m, bm), alpha = m == -INFINITY ? 0.f : expf(m - m_new);
                m = m_new;
                l *= alpha;
#pragma unroll
                for (int i = 0; i < DT; ++i) acc[i] *= alpha;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sc[j] = sc[j] == -INFINITY ? 0.f : expf(sc[j] - m);
                l += sc[j];
            }
            // values of keys that do not exist (behind the request's end, in a page that is gone) may be anything
#pragma unroll
            for (int i = 0; i < DT; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[i][j] = j < n_ok ? v[i][j] : 0.f;
            // A key that some rows read and others do not has weight zero for these, which takes no infinity and no NaN away:
            // a block with both goes key by key, each row by its own keys
            bool odd = false;
            if (__any(hidden)) {
                af_f32x4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < DT; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) z[j] = fmaf(v[i][j], 0.f, z[j]);
                odd = __any(!(z[0] + z[1] + z[2] + z[3] == 0.f));
            }
            if (!odd) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < DT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i][j], sc[j], acc[i], 0, 0, 0);
            } else {
#pragma unroll 1
                for (int kg = 0; kg < 4; ++kg)                                             // (lane kg of a group of four has its keys)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int key = lo + 16 * b + 4 * kg + j;
                        const bool reads = key <= pos && key >= first && page_ok;
                        const float w = __shfl(sc[j], 16 * kg + r, 64);
#pragma unroll
                        for (int i = 0; i < DT; ++i)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float x = __shfl(v[i][j], 16 * kg + 4 * g + e, 64);
                                if (reads) acc[i][e] = fmaf(w, x, acc[i][e]);
                            }
                    }
            }
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    // lane (row r, g) has dims 16 i + 4 g .. of its row; the waves meet in LDS, wave w then has the dims of i = w, w + AF ..
#pragma unroll
    for (int i = 0; i < DT; ++i) *reinterpret_cast<af_f32x4_t*>(lo_[wave][i][lane]) = acc[i];
    if (g == 0) { lm_[wave][r] = m; ll_[wave][r] = l; }
    __syncthreads();
    float M = lm_[0][r];
#pragma unroll
    for (int w = 1; w < AF; ++w) M = fmaxf(M, lm_[w][r]);
    float wt[AF], L = 0.f;
#pragma unroll
    for (int w = 0; w < AF; ++w) {
        wt[w] = lm_[w][r] == -INFINITY ? 0.f : expf(lm_[w][r] - M);
        L += ll_[w][r] * wt[w];
    }
    if (!row_ok) return;
    float* part = a.ws + (((size_t)tile * a.n_kv + hk) * a.splits + sp) * 16 * (D + 2);
#pragma unroll
    for (int i = wave; i < DT; i += AF) {
        af_f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < AF; ++w) o += wt[w] * *reinterpret_cast<const af_f32x4_t*>(lo_[w][i][lane]);
        if (a.splits > 1) *reinterpret_cast<af_f32x4_t*>(part + r * D + 16 * i + 4 * g) = o;
        else af_store(a, q0 + tq, head * D + 16 * i + 4 * g, a.n_q * D, o, L);
    }
    if (a.splits > 1 && wave == 0 && g == 0) { part[16 * D + r] = M; part[16 * D + 16 + r] = L; }
}

// The parts of a (tile, kv head) added in their order: one block, thread (row, four dims) in turn.
template <int D>
__global__ __launch_bounds__(256) void attention_f32_merge_kernel(AfArgs a) {
    const int hk = blockIdx.x, tile = blockIdx.y, G = a.n_q / a.n_kv;
    const int s = a.tile_entry[tile], row0 = a.tile_row0[tile], q0 = a.cu_q[s], nrows = (a.cu_q[s + 1] - q0) * G;
    const float* base = a.ws + ((size_t)tile * a.n_kv + hk) * a.splits * 16 * (D + 2);
    for (int e = threadIdx.x; e < 16 * (D / 4); e += 256) {
        const int r = e / (D / 4), c = (e % (D / 4)) * 4, row = row0 + r;
        if (row >= nrows) continue;
        float M = -INFINITY, L = 0.f;
        for (int i = 0; i < a.splits; ++i) M = fmaxf(M, base[(size_t)i * 16 * (D + 2) + 16 * D + r]);
        af_f32x4_t o = {0.f, 0.f, 0.f, 0.f};
        for (int i = 0; i < a.splits; ++i) {
            const float* p = base + (size_t)i * 16 * (D + 2);
            const float mi = p[16 * D + r], w = mi == -INFINITY ? 0.f : expf(mi - M);
            L += p[16 * D + 16 + r] * w;
            o += w * *reinterpret_cast<const af_f32x4_t*>(p + r * D + c);
        }
        af_store(a, q0 + row / G, (hk * G + row % G) * D + c, a.n_q * D, o, L);
    }
}

// floats of workspace for `splits` > 1 parts
extern "C" int64_t spy_attention_f32_workspace(int tiles, int n_kv, int d, int splits) {
    return splits > 1 ? (int64_t)tiles * n_kv * splits * 16 * (d + 2) : 0;
}

extern "C" int spy_attention_f32(float* out, const float* q, const float* kc, const float* vc, int P, int num_pages, const int* cu_q,
                                 const int* pos0, const int* kv_len, const int* block_table, int max_blocks, const int* tile_entry,
                                 const int* tile_row0, int tiles, int S, int T, int n_q, int n_kv, int d, float scale, int window,
                                 float softcap, int splits, float* ws, const float* raw_qkv, const float* qw, const float* kw, float eps,
                                 const float* cos_t, const float* sin_t, int max_pos, int store, const float* dist, const float* sink, int chunk,
                                 const float* gate, long long gate_ld, hipStream_t st) {
    SPY_REQUIRE(T > 0 && S > 0 && n_q > 0 && n_kv > 0 && P > 0 && num_pages > 0 && max_blocks > 0 && tiles > 0, "spy_attention_f32: empty operand");
    SPY_REQUIRE((d == 64 || d == 128) && P % 16 == 0, "spy_attention_f32: head_dim %d and pages of %d are not for this kernel", d, P);
    SPY_REQUIRE(n_q % n_kv == 0 && tiles <= 65535 && splits >= 1 && splits <= 64, "spy_attention_f32: %d tiles of %d / %d heads in %d parts", tiles, n_q, n_kv, splits);
    SPY_REQUIRE(splits == 1 || ws, "spy_attention_f32: no workspace");
    SPY_REQUIRE(chunk >= 0 && !(chunk > 0 && window > 0), "spy_attention_f32: a window or chunks, not both");
    SPY_REQUIRE(!gate || gate_ld >= (long long)n_q * d, "spy_attention_f32: the gate's rows are too short");
    const uintptr_t at = (uintptr_t)out | (uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc | (uintptr_t)ws;
    SPY_REQUIRE(at % 16 == 0, "spy_attention_f32: operands must be 16-byte aligned");
    const AfArgs a = {out, q, kc, vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, tile_entry, tile_row0, n_q, n_kv,
                      scale, window, softcap, splits, ws, dist, sink, chunk, gate, gate_ld};
    const dim3 grid(n_kv, tiles, splits);
    if (raw_qkv) {
        const uintptr_t raw = (uintptr_t)raw_qkv | (uintptr_t)qw | (uintptr_t)kw | (uintptr_t)cos_t | (uintptr_t)sin_t;
        SPY_REQUIRE(raw % 16 == 0 && (qw == nullptr) == (kw == nullptr) && (cos_t == nullptr) == (sin_t == nullptr) && (!cos_t || max_pos > 0),
                    "spy_attention_f32: operands of the raw product");
        SPY_REQUIRE(tiles == S && T == S && n_q / n_kv <= 16 && !gate && !dist && !sink && !chunk && softcap == 0.f, "spy_attention_f32: the raw product is for single tokens");
        const AfRaw z = {raw_qkv, qw, kw, eps, cos_t, sin_t, max_pos, store};
        if (d == 64) attention_f32_kernel<64, true><<<grid, AF * 64, 0, st>>>(a, tiles, z);
        else attention_f32_kernel<128, true><<<grid, AF * 64, 0, st>>>(a, tiles, z);
    } else {
        if (d == 64) attention_f32_kernel<64, false><<<grid, AF * 64, 0, st>>>(a, tiles, AfRaw{});
        else attention_f32_kernel<128, false><<<grid, AF * 64, 0, st>>>(a, tiles, AfRaw{});
    }
    SPY_CHECK_LAUNCH("spy_attention_f32");
    if (splits > 1) {
        if (d == 64) attention_f32_merge_kernel<64><<<dim3(n_kv, tiles), 256, 0, st>>>(a);
        else attention_f32_merge_kernel<128><<<dim3(n_kv, tiles), 256, 0, st>>>(a);
        SPY_CHECK_LAUNCH("spy_attention_f32 (merge)");
    }
    return 0;
}
