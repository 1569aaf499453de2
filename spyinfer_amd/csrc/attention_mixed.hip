// Attention of a step that has entries with many query rows beside entries with few (a portion of a prompt beside requests
// that decode, long prompts beside short ones) in one launch of blocks of eight waves: the first `big` blocks take 128-row
// tiles (attention_tiles.h), the others a 16-row tile and a kv head each, the eight waves its keys in turn (attention_rows.h).
//
// Each kind of its own is bound by its longest block, not by the chip: a chain of rounds of 64 keys, or of turns of the
// waves, on a part of the compute units.  Apart they run one after the other; here they run beside each other, and the
// second launch and the gap before it are saved.
#include "attention_rows.h"
#include "attention_tiles.h"

template <int DMAX, int FULL>
__global__ __launch_bounds__(512, 2) void attention_mixed_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, bf16_t* kc, bf16_t* vc, int P, int num_pages, const int* __restrict__ cu_q,
    const int* __restrict__ pos0, const int* __restrict__ kv_len, const int* __restrict__ block_table, int max_blocks,
    const int* __restrict__ big_entry, const int* __restrict__ big_row0, int num_big, const int* __restrict__ small_entry,
    const int* __restrict__ small_row0, int n_q, int n_kv, float scale, int window, float softcap, int log2p, int out_tiles,
    const float* __restrict__ dist, const float* __restrict__ sink, int chunk, OutGate og, int paired, int gx) {
    constexpr int KS = PF_KEYS * (DMAX + 16), VS = DMAX * (PF_KEYS + 16);
    __shared__ __attribute__((aligned(16))) bf16_t lds[KS + VS];
    static_assert(sizeof(lds) >= AW * (DMAX / 16 * 4 + 2) * 64 * sizeof(float), "the waves' sums fit where the keys and values are staged");
    const int big = gx * n_kv, b = blockIdx.x;
    if (b < big) {
        attention_prefill_body<DMAX, true, 1, 128>(out, q, kc, vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, big_entry, big_row0,
                                                   n_q, n_kv, DMAX, scale, window, softcap, log2p, num_big, 1, nullptr, out_tiles, dist, sink,
                                                   chunk, og, paired, b, gx, n_kv, 1, lds, lds + KS);
    } else {
        const FusedQKV none = {};
        attention_mfma_body<DMAX, false, FULL, 2 * AW>(out, q, kc, vc, P, num_pages, cu_q, pos0, kv_len, block_table, max_blocks, small_entry,
                                                       small_row0, n_q, n_kv, DMAX, scale, window, softcap, 1, nullptr, none, out_tiles, nullptr,
                                                       log2p, nullptr, dist, sink, chunk, og, (b - big) / n_kv, (b - big) % n_kv, 0,
                                                       reinterpret_cast<float*>(lds));
    }
}

// Both kinds of tiles, each with all of its keys in one part; head sizes 64 and 128, pages of a power of two.  out_tiles: as
// for spy_attention_prefill.
extern "C" int spy_attention_mixed(void* out, const void* q, void* kc, void* vc, int P, int num_pages, const int* cu_q, const int* pos0,
                                   const int* kv_len, const int* block_table, int max_blocks, const int* big_entry, const int* big_row0,
                                   int num_big, const int* small_entry, const int* small_row0, int num_small, int S, int T, int n_q, int n_kv,
                                   int d, float scale, int window, float softcap, int out_tiles, const float* dist, const float* sink, int chunk,
                                   const void* gate, long long gate_ld, hipStream_t st) {
    SPY_REQUIRE(num_big > 0 && num_small > 0 && S > 0 && T > 0 && n_q > 0 && n_kv > 0 && num_pages > 0 && max_blocks > 0,
                "spy_attention_mixed: empty operand");
    SPY_REQUIRE(d == 64 || d == 128, "spy_attention_mixed: head_dim %d (64 or 128 allowed)", d);
    SPY_REQUIRE(P >= 8 && (P & (P - 1)) == 0, "spy_attention_mixed: page size %d is not a power of two >= 8", P);
    SPY_REQUIRE(n_q % n_kv == 0, "spy_attention_mixed: n_q %d is not a multiple of n_kv %d", n_q, n_kv);
    SPY_REQUIRE(out_tiles >= 0 && out_tiles <= 8 && (!out_tiles || (T <= 16 * out_tiles && (n_q * d) % 32 == 0)),
                "spy_attention_mixed: operand order is for at most 128 rows (%d here) of a width that is a multiple of 32", T);
    SPY_REQUIRE(softcap >= 0.f && chunk >= 0 && !(chunk > 0 && window > 0), "spy_attention_mixed: a window or chunks, not both, and no negative cap");
    SPY_REQUIRE(!gate || (gate_ld >= (long long)n_q * d && gate_ld % 4 == 0 && ((uintptr_t)gate % 8) == 0),
                "spy_attention_mixed: the gate's rows are too short or not aligned");
    const OutGate og = {(const bf16_t*)gate, gate_ld};
    int log2p = 0;
    while ((1 << log2p) < P) ++log2p;
    const long long cus = attention_compute_units();
    const bool paired = (long long)num_big * n_kv > cus;          // (as in spy_attention_prefill)
    const int gx = paired ? (num_big + 1) / 2 : num_big;
    const long long blocks = ((long long)gx + num_small) * n_kv;
    SPY_REQUIRE(blocks <= 0x7fffffff, "spy_attention_mixed: too many blocks");
#define AX_LAUNCH(DM, FL)                                                                                                          \
    attention_mixed_kernel<DM, FL><<<(unsigned)blocks, 512, 0, st>>>((bf16_t*)out, (const bf16_t*)q, (bf16_t*)kc, (bf16_t*)vc, P,  \
        num_pages, cu_q, pos0, kv_len, block_table, max_blocks, big_entry, big_row0, num_big, small_entry, small_row0, n_q, n_kv,  \
        scale, window, softcap, log2p, out_tiles, dist, sink, chunk, og, paired, gx)
    if (d == 64) { if (P <= 32) AX_LAUNCH(64, FULL_STREAMED); else AX_LAUNCH(64, FULL_KEPT); }
    else if (P <= 32) AX_LAUNCH(128, FULL_STREAMED);
    else AX_LAUNCH(128, FULL_KEPT);
#undef AX_LAUNCH
    SPY_CHECK_LAUNCH("spy_attention_mixed");
    return 0;
}
