// Paged attention on MFMA for entries with many query rows: the launches (the kernel's body, and what it does, is
// attention_tiles.h).
#include "attention_tiles.h"

// MINW: waves per SIMD that the registers must allow.  The 8-wave shape with 4 (128 registers, two blocks per CU) is
// the fastest shape for grids of more than one block per CU; with one block per CU it is 6 % faster with the
// registers of 2.
template <int DMAX, bool DFULL, int RT, int MINW, int PF_ROWS>
__global__ __launch_bounds__(PF_ROWS / RT * 4, MINW) void attention_prefill_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    int P, int num_pages, const int* __restrict__ cu_q, const int* __restrict__ pos0, const int* __restrict__ kv_len,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tile_entry, const int* __restrict__ tile_row0,
    int n_q, int n_kv, int d, float scale, int window, float softcap, int log2p, int num_tiles, int splits, float* __restrict__ ws, int out_tiles,
    const float* __restrict__ dist, const float* __restrict__ sink, int chunk, OutGate og, int paired) {
    __shared__ __attribute__((aligned(16))) bf16_t ks[PF_KEYS * (DMAX + 16)];
    __shared__ __attribute__((aligned(16))) bf16_t vs[DMAX * (PF_KEYS + 16)];
    const int gx = gridDim.x, gy = gridDim.y, lin = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    attention_prefill_body<DMAX, DFULL, RT, PF_ROWS>(out, q, kc, vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, tile_entry,
                                                     tile_row0, n_q, n_kv, d, scale, window, softcap, log2p, num_tiles, splits, ws, out_tiles,
                                                     dist, sink, chunk, og, paired, lin, gx, gy, gridDim.z, ks, vs);
}

extern "C" int64_t spy_attention_prefill_workspace(int num_tiles, int tile_rows, int n_kv, int d, int splits) {
    if (splits <= 1) return 0;
    return (int64_t)num_tiles * (tile_rows / 16) * n_kv * splits * 16 * ((d <= 64 ? 64 : 128) + 2);
}

// Tiles of 256 rows against tiles of 128, same measurement: 92 against 73 us at 2048 tokens (128 blocks: half the CUs
// idle), 125 against 133 at 3072, 170 against 195 at 4096, 607 against 675 at 8192, 2331 against 2565 at 16384 (0.94
// PFLOP/s); the caller picks the tile size by the number of blocks.  One tile per block instead of two, so that a grid
// of one block per CU becomes two per CU, was slower at every length (88 against 73 us at 2048 tokens); where one tile per
// block leaves every block a CU of its own it is the faster way: 12.0 against 19.0 us at 100 tokens (32 tiles), 19.6 against
// 26.6 at 389 (104), 30.7 against 36.9 at 800 (200), 35.9 against 41.8 at 1000 (256), 17.8 against 24.5 for two prompts of 300.
// Measured on MI355X (256 CUs), 32 query heads of 128, microseconds per call for 2048 / 2304 / 3072 / 4096 / 8192
// tokens of one prompt (256 / 288 / 384 / 512 / 1024 blocks): 4 waves of two row tiles 85 / 115 / 148 / 193 / 717;
// 8 waves of one row tile with registers for one block per CU 65 / 130 / 165 / 217 / 807, with 128 registers (two
// blocks per CU) 69 / 98 / 129 / 185 / 677.  So: 8 waves always (full head sizes), the registers by the grid.
extern "C" int spy_attention_prefill(void* out, const void* q, const void* kc, const void* vc, int P, int num_pages, const int* cu_q,
                                     const int* pos0, const int* kv_len, const int* block_table, int max_blocks,
                                     const int* tile_entry, const int* tile_row0, int num_tiles, int tile_rows, int S, int T, int n_q,
                                     int n_kv, int d, float scale, int window, float softcap, int splits, float* ws, int out_tiles, const float* dist, const float* sink,
                                     int chunk, const void* gate, long long gate_ld, hipStream_t st) {
    SPY_REQUIRE(num_tiles > 0 && S > 0 && T > 0 && n_q > 0 && n_kv > 0 && num_pages > 0 && max_blocks > 0,
                "spy_attention_prefill: empty operand");
    SPY_REQUIRE(d % 16 == 0 && d >= 16 && d <= 128, "spy_attention_prefill: head_dim %d is not a multiple of 16 in 16..128", d);
    SPY_REQUIRE(P >= 8 && (P & (P - 1)) == 0, "spy_attention_prefill: page size %d is not a power of two >= 8", P);
    int log2p = 0;
    while ((1 << log2p) < P) ++log2p;
    SPY_REQUIRE(n_q % n_kv == 0, "spy_attention_prefill: n_q %d is not a multiple of n_kv %d", n_q, n_kv);
    SPY_REQUIRE(n_kv <= 65535, "spy_attention_prefill: too many kv heads");
    SPY_REQUIRE(splits >= 1 && splits <= 16, "spy_attention_prefill: %d key parts (1..16 allowed)", splits);
    SPY_REQUIRE(splits == 1 || ws, "spy_attention_prefill: key parts without a workspace");
    SPY_REQUIRE(tile_rows == 128 || (tile_rows == 256 && (d == 64 || d == 128)),
                "spy_attention_prefill: tiles of %d rows (128, or 256 for head sizes 64 and 128)", tile_rows);
    // out_tiles > 0: the output [T, n_q d] goes out in MFMA operand order for that many row tiles (attention_merge.h), for a
    // decode product that reads it next
    SPY_REQUIRE(out_tiles >= 0 && out_tiles <= 8 && (!out_tiles || (T <= 16 * out_tiles && (n_q * d) % 32 == 0 && d % 8 == 0)),
                "spy_attention_prefill: operand order is for at most 128 rows (%d here) of a width that is a multiple of 32", T);
    SPY_REQUIRE(chunk >= 0 && !(chunk > 0 && window > 0), "spy_attention_prefill: a window or chunks, not both");
    SPY_REQUIRE(!gate || (gate_ld >= (long long)n_q * d && gate_ld % 4 == 0 && ((uintptr_t)gate % 8) == 0),
                "spy_attention_prefill: the gate's rows are too short or not aligned");
    const OutGate og = {(const bf16_t*)gate, gate_ld};
    const bool paired = splits == 1 && (long long)num_tiles * n_kv > attention_compute_units();
    const dim3 grid(paired ? (num_tiles + 1) / 2 : num_tiles, n_kv, splits);
    const dim3 mgrid(num_tiles * (tile_rows / 16), n_kv);
    const bool one_per_cu = (long long)grid.x * grid.y * grid.z <= attention_compute_units();
#define PF_ARGS (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc, P, num_pages, cu_q, pos0, kv_len, block_table,   \
                max_blocks, tile_entry, tile_row0, n_q, n_kv, d, scale, window, softcap, log2p, num_tiles, splits, ws, out_tiles, dist, sink, \
                chunk, og, paired
    // (head sizes other than 64 and 128 keep the 4-wave shape: with conditions in the head-dim loops the other needs too many registers)
#define PF_CASE(DM)                                                                                                              \
    if (tile_rows == 256) attention_prefill_kernel<DM, true, 2, 2, 256><<<grid, 512, 0, st>>>(PF_ARGS);                          \
    else if (d == DM) {                                                                                                          \
        if (one_per_cu) attention_prefill_kernel<DM, true, 1, 2, 128><<<grid, 512, 0, st>>>(PF_ARGS);                            \
        else attention_prefill_kernel<DM, true, 1, 4, 128><<<grid, 512, 0, st>>>(PF_ARGS);                                       \
    } else attention_prefill_kernel<DM, false, 2, 2, 128><<<grid, 256, 0, st>>>(PF_ARGS);                                        \
    if (splits > 1)                                                                                                              \
        attention_merge_kernel<DM><<<mgrid, 256, 0, st>>>((bf16_t*)out, ws, cu_q, tile_entry, tile_row0, n_q, n_kv, d, splits,    \
                                                          tile_rows / 16, out_tiles, og);
    if (d <= 64) { PF_CASE(64) } else { PF_CASE(128) }
#undef PF_CASE
#undef PF_ARGS
    SPY_CHECK_LAUNCH("spy_attention_prefill");
    return 0;
}
