// The gated delta rule over chunks of 16 tokens through the matrix cores (delta_chunks.hip), for steps that hold more than single tokens.
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

bool delta_chunks_takes(int S, int T, int d, int dv);
int64_t delta_chunks_workspace(int S, int T, int H, int d, int dv);
int delta_chunks(const DeltaChunks& a, int dtype, hipStream_t st);
