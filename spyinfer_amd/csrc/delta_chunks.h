// The gated delta rule and the mLSTM over chunks of 16 tokens through the matrix cores (delta_chunks.hip), for steps that hold more than
// single tokens.
#pragma once
#include "common.h"

struct DeltaChunks {
    float* o;                // [T, H dv] the read-outs
    float* state;
    long long state_stride;
    const void* qkv;         // [T, 2 G d + H dv]: v behind q and k
    const float* qk;         // [T, 2 G d] unit vectors
    const float* beta;       // sigmoid'ed, rows bs apart
    const float* dec;        // decays, rows zs apart
    const int* cu_q;
    const int* slot_ids;
    int num_slots, S, T, H, G, d, dv, dd;
    long long bs, zs;
    float* ws;
    int64_t ws_floats;
};

// The mLSTM's matrix memory by the same chunks: S = a S + b k v^T, n = a n + b k, o = S^T q / (max(|n . q|, e^-m) + 1e-6) with a, b and
// e^-m known for every token (abe [T, 3 H]) and the entries' last maxima in mfin [S, H].
struct MemoryChunks {
    float* o;                // [T, H dv] the read-outs
    float* state;            // a request's: per head S [d, dv], then per slice of 16 channels n [d] and m
    const void* x;           // rows xs apart: q at q_off, k at k_off (H heads of d), v at v_off (H heads of dv)
    long long xs;
    int q_off, k_off, v_off;
    const float* abe;
    const float* mfin;
    const int* cu_q;
    const int* slot_ids;
    int num_slots, S, T, H, d, dv;
    float* ws;
    int64_t ws_floats;
};

bool delta_chunks_takes(int S, int T, int d, int dv);
int64_t delta_chunks_workspace(int S, int T, int H, int d, int dv);
int delta_chunks(const DeltaChunks& a, int dtype, hipStream_t st);
int memory_chunks(const MemoryChunks& a, int dtype, hipStream_t st);
