// Grouped expert products of a MoE prefill chunk with few tokens per expert
// (moe_stream.hip); the tile list and the rest of the chunk are in prefill.hip.
#pragma once

#include "common.h"

namespace gdsllm {

struct MoeStreamArgs {
    const uint8_t* w;   // affine words of the stacked pool (dual: gate)
    const uint8_t* s;
    const uint8_t* b;
    const uint8_t* w2;  // dual: up
    const uint8_t* s2;
    const uint8_t* b2;
    int64_t estride_w, estride_s, estride_b;  // per-expert byte strides
    const uint16_t* x;
    uint16_t* y;
    int M, K;           // output rows, columns of one expert matrix
    int64_t ldx, ldy;
    const int4* tiles;  // (expert, p0, n, 0) on the device, n <= 2 kStreamTokens, two-pass ones first
    const int* passes;  // passes of at most kStreamTokens positions, then the number of two-pass tiles
    const int* tok;     // X row of each position, or null: X rows are the positions
};

constexpr int kStreamTokens = 16;  // positions of one pass over an expert's rows

// Whether moe_stream serves expert matrices of M rows x K columns.
bool moe_stream_fits(int64_t M, int64_t K);
// Workgroups per pass over an expert matrix of M rows.
int moe_stream_jobs(int64_t M, bool dual);
// y[p][r] = x[tok[p]] . W_e[r] for the positions p of at most max_passes passes
// over expert e; dual: fp16(silu(gate) * up) of the two pools.  group_size 32,
// 64 or 128; arguments already validated.
int moe_stream(const MoeStreamArgs& a, int group_size, bool dual, int64_t max_passes, hipStream_t stream);

}  // namespace gdsllm
