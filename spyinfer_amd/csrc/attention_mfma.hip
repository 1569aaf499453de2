// Paged attention on MFMA over 16-row tiles: the launches (the kernel's body, and what it does, is attention_rows.h).
#include "attention_rows.h"

template <int DMAX, bool FUSED, int FULL>
__global__ __launch_bounds__(AW * 64, (FUSED && DMAX <= 128) ? 2 : 1) void attention_mfma_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, bf16_t* kc, bf16_t* vc,
    int P, int num_pages, const int* __restrict__ cu_q, const int* __restrict__ pos0, const int* __restrict__ kv_len,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tile_entry, const int* __restrict__ tile_row0,
    int n_q, int n_kv, int d, float scale, int window, float softcap, int splits, float* __restrict__ ws, FusedQKV fz, int out_tiles,
    unsigned* counters, int log2p, const int* __restrict__ pieces, const float* __restrict__ dist,
    const float* __restrict__ sink, int chunk, OutGate og) {
    extern __shared__ float lds[];
    attention_mfma_body<DMAX, FUSED, FULL>(out, q, kc, vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, tile_entry, tile_row0,
                                           n_q, n_kv, d, scale, window, softcap, splits, ws, fz, out_tiles, counters, log2p, pieces, dist,
                                           sink, chunk, og, blockIdx.x, blockIdx.y, blockIdx.z, lds);
}

// The fused variant by blocks of eight waves (heads of 128), one a compute unit: for steps that have no more blocks than units.  A block's
// waves then have half the turns, and the unit as many loads under way as with two blocks of four.  Two blocks of keys a wave under way, in two sets of registers,
// were 0.8 us slower a launch (25 KB of code for 16).  Where the line lies: piece_waves in kernels/key_pieces.py.
template <int FULL>
__global__ __launch_bounds__(2 * AW * 64, 1) void attention_mfma_wide_kernel(
    bf16_t* __restrict__ out, bf16_t* kc, bf16_t* vc,
    int P, int num_pages, const int* __restrict__ cu_q, const int* __restrict__ pos0, const int* __restrict__ kv_len,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tile_entry, const int* __restrict__ tile_row0,
    int n_q, int n_kv, float scale, int window, float* __restrict__ ws, FusedQKV fz, int out_tiles, unsigned* counters, int log2p,
    const int* __restrict__ pieces) {
    __shared__ float lds[2 * AW * (128 / 4 + 2) * 64];
    attention_mfma_body<128, true, FULL, 2 * AW>(out, nullptr, kc, vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, tile_entry, tile_row0,
                                                 n_q, n_kv, 128, scale, window, 0.f, 1, ws, fz, out_tiles, counters, log2p, pieces, nullptr,
                                                 nullptr, 0, OutGate{}, blockIdx.x, blockIdx.y, blockIdx.z, lds);
}

static int dmax_of(int d) { return d <= 64 ? 64 : (d <= 128 ? 128 : 256); }

// Floats of one part's sums in the workspace (keys cut by the host: one part per record).
extern "C" int64_t spy_attention_mfma_part_workspace(int d) { return 16 * (dmax_of(d) + 2); }

extern "C" int64_t spy_attention_mfma_workspace(int num_tiles, int n_kv, int d, int splits) {
    if (splits <= 1) return 0;
    return (int64_t)num_tiles * n_kv * splits * 16 * (dmax_of(d) + 2);
}

// out_tiles > 0: the output [T, n_q d] goes out in MFMA operand order for that many row tiles (attention_merge.h), for a
// decode product that reads it next.
// qkv != null: the fused variant (see the top of the file).  Then q is not read, every entry must be a single token
// (T == S), head_dim 64, 128 or 256 with the whole head rotated (or no rotation: cos_t == null), and the new keys and
// values are written to kc and vc by this call (store != 0).  waves: of a block, 4, or 8 for keys cut by the host and heads of 128.
extern "C" int spy_attention_mfma(void* out, const void* q, void* kc, void* vc, int P, int num_pages, const int* cu_q,
                                  const int* pos0, const int* kv_len, const int* block_table, int max_blocks, const int* tile_entry,
                                  const int* tile_row0, int num_tiles, int S, int T, int n_q, int n_kv, int d, float scale,
                                  int window, float softcap, int splits, float* ws, const void* qkv, const void* qw, const void* kw, int w_dtype,
                                  float eps, const float* cos_t, const float* sin_t, int max_pos, int store, int out_tiles,
                                  unsigned* counters, int n_counters, const int* pieces, int num_pieces, const float* dist, const float* sink,
                                  int chunk, const void* gate, long long gate_ld, int waves, hipStream_t st) {
    SPY_REQUIRE(!qkv || (!dist && !sink && !gate && !chunk), "spy_attention_mfma: the fused variant takes neither a penalty on the distance nor a sink, chunks or a gate");
    SPY_REQUIRE(chunk >= 0 && !(chunk > 0 && window > 0), "spy_attention_mfma: a window or chunks, not both");
    SPY_REQUIRE(!gate || (gate_ld >= (long long)n_q * d && gate_ld % 4 == 0 && ((uintptr_t)gate % 8) == 0),
                "spy_attention_mfma: the gate's rows are too short or not aligned");
    const OutGate og = {(const bf16_t*)gate, gate_ld};
    SPY_REQUIRE(num_tiles > 0 && S > 0 && T > 0 && n_q > 0 && n_kv > 0 && num_pages > 0 && max_blocks > 0,
                "spy_attention_mfma: empty operand");
    SPY_REQUIRE(d % 16 == 0 && d >= 16 && d <= 256, "spy_attention_mfma: head_dim %d is not a multiple of 16 in 16..256", d);
    SPY_REQUIRE(P % 8 == 0, "spy_attention_mfma: page size %d is not a multiple of 8", P);
    SPY_REQUIRE(n_q % n_kv == 0, "spy_attention_mfma: n_q %d is not a multiple of n_kv %d", n_q, n_kv);
    SPY_REQUIRE(splits >= 1 && splits <= 64, "spy_attention_mfma: %d parts (1..64 allowed)", splits);
    SPY_REQUIRE(splits == 1 || ws, "spy_attention_mfma: parts without a workspace");
    SPY_REQUIRE(n_kv <= 65535, "spy_attention_mfma: too many kv heads");
    SPY_REQUIRE(out_tiles >= 0 && out_tiles <= 8 && (!out_tiles || (T <= 16 * out_tiles && (n_q * d) % 32 == 0 && d % 8 == 0)),
                "spy_attention_mfma: operand order is for at most 128 rows (%d here) of a width that is a multiple of 32", T);
    SPY_REQUIRE(softcap >= 0.f && (!qkv || softcap == 0.f), "spy_attention_mfma: the scores' cap must not be negative, and the fused variant takes none");
    FusedQKV fz = {(const bf16_t*)qkv, qw, kw, w_dtype, eps, cos_t, sin_t, max_pos, store};
    if (qkv) {
        SPY_REQUIRE(T == S && num_tiles == S, "spy_attention_mfma: the fused variant takes single tokens only (%d tokens of %d entries)", T, S);
        SPY_REQUIRE(d == 64 || d == 128 || d == 256, "spy_attention_mfma: the fused variant takes head_dim 64, 128 or 256, not %d", d);
        SPY_REQUIRE((!cos_t) == (!sin_t) && (!cos_t || max_pos > 0), "spy_attention_mfma: rotation tables are incomplete");
        SPY_REQUIRE((!qw) == (!kw) && (!qw || w_dtype == SPY_F32 || w_dtype == SPY_BF16), "spy_attention_mfma: norm weights are incomplete");
        SPY_REQUIRE(n_q / n_kv <= 16, "spy_attention_mfma: the fused variant takes groups of at most 16 heads");
        SPY_REQUIRE(((uintptr_t)qkv % 16) == 0, "spy_attention_mfma: qkv must be 16-byte aligned");
    } else {
        SPY_REQUIRE(q, "spy_attention_mfma: no queries");
    }
    if (pieces) {
        // the keys cut by the host (see the kernel's top): one block per record, parts merged by their last block only
        SPY_REQUIRE(qkv && num_pieces > 0, "spy_attention_mfma: keys cut by the host are for the fused variant");
        SPY_REQUIRE(d <= 128 && counters && ws && (long long)num_tiles * n_kv <= n_counters && ((uintptr_t)pieces % 16) == 0,
                    "spy_attention_mfma: keys cut by the host need head_dim <= 128, a workspace and a counter per (entry, kv head) (%d x %d, %d counters)",
                    num_tiles, n_kv, n_counters);
    }
    int log2p = -1;                                        // pages of a power of two: shifts instead of divisions
    if ((P & (P - 1)) == 0) { log2p = 0; while ((1 << log2p) < P) ++log2p; }
    const dim3 grid = pieces ? dim3(num_pieces, 1, 1) : dim3(num_tiles, n_kv, splits);
    const dim3 mgrid(num_tiles, n_kv);
    SPY_REQUIRE(waves == AW || (waves == 2 * AW && pieces && d == 128), "spy_attention_mfma: blocks of %d waves", waves);
    if (waves == 2 * AW) {
#define ATT_WIDE(FL)                                                                                                          \
        attention_mfma_wide_kernel<FL><<<grid, 2 * AW * 64, 0, st>>>((bf16_t*)out, (bf16_t*)kc, (bf16_t*)vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, \
                                                                     tile_entry, tile_row0, n_q, n_kv, scale, window, ws, fz, out_tiles, counters, log2p, pieces)
        if (P <= 32) ATT_WIDE(FULL_STREAMED); else ATT_WIDE(FULL_KEPT);
#undef ATT_WIDE
        SPY_CHECK_LAUNCH("spy_attention_mfma");
        return 0;
    }
    // The parts merged by each (tile, kv head)'s last block instead of a second kernel: with counters (zeroed once by the
    // caller, one per tile and head, left at zero by every call; calls that overlap on one device race on them), up to
    // 16 parts (the grid's; the host's records may name up to 32 of an entry) and head sizes up to 128.
    unsigned* const cnt = (pieces || (counters && splits > 1 && splits <= 16 && d <= 128 && (long long)num_tiles * n_kv <= n_counters)) ? counters : nullptr;
#define ATT_LAUNCH(DM, FZ, FL)                                                                                                \
    attention_mfma_kernel<DM, FZ, FL><<<grid, AW * 64, (DM <= 128 ? AW : AW - 1) * ((DM / 16) * 4 + 2) * 64 * sizeof(float), st>>>(  \
        (bf16_t*)out, (const bf16_t*)q, (bf16_t*)kc, (bf16_t*)vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks,  \
        tile_entry, tile_row0, n_q, n_kv, d, scale, window, softcap, splits, ws, fz, out_tiles, cnt, log2p, pieces, dist, sink, chunk, og)
#define ATT_CASE(DM)                                                                                                          \
    if (qkv && P <= 32) ATT_LAUNCH(DM, true, FULL_STREAMED); else if (qkv) ATT_LAUNCH(DM, true, FULL_KEPT);                      \
    else if (d == DM && P <= 32) ATT_LAUNCH(DM, false, FULL_STREAMED); else if (d == DM) ATT_LAUNCH(DM, false, FULL_KEPT);       \
    else ATT_LAUNCH(DM, false, 0);                                                                                            \
    if (cnt) {}                                                                                                               \
    else if (splits > 1 && qkv)                                                                                               \
        attention_merge_kernel<DM, true><<<mgrid, 256, 0, st>>>((bf16_t*)out, ws, cu_q, tile_entry, tile_row0, n_q, n_kv, d, splits, 1, out_tiles); \
    else if (splits > 1)                                                                                                      \
        attention_merge_kernel<DM><<<mgrid, 256, 0, st>>>((bf16_t*)out, ws, cu_q, tile_entry, tile_row0, n_q, n_kv, d, splits, 1, out_tiles, og);
    switch (dmax_of(d)) {
        case 64: ATT_CASE(64) break;
        case 128: ATT_CASE(128) break;
        default: ATT_CASE(256) break;
    }
#undef ATT_CASE
#undef ATT_LAUNCH
    SPY_CHECK_LAUNCH("spy_attention_mfma");
    return 0;
}
