// Parameters of a linear product, as the kernels take them.
#pragma once

#include "common.h"

namespace flux {

struct GemmParams {
    const bf16_t* A; const bf16_t* W; const bf16_t* bias;
    bf16_t* Y; bf16_t* Y2;
    const bf16_t* resid; const bf16_t* gate;
    int M, N, K;
    int a_rows;          // A's rows come in batches of this many ...
    int64_t a_skip;      // ... with this many elements beyond lda between two batches (0: evenly strided)
    int64_t lda, ldw, ldy, ldy2, ldresid, gate_stride;
    int split_n, y2_col0, rows_per_batch;
    int act, act_begin;
    int in_silu;  // 1: A passes through x * sigmoid(x), rounded to bf16, on the way in (row-vector and scalar kernels)
    int bias_vec;  // 1: bias may be read with 8-byte buffer loads (4-byte aligned base)
    int vec_io;  // 1: every output/residual row segment of 8 columns may be accessed as 16 bytes
    int checked; // 1: an eight-wave tile takes the epilogue that decides per column
    // fused QK RMSNorm + RoPE for columns [0, qk_cols): q heads first, then k heads, 128 columns each
    bf16_t* q_out; bf16_t* k_out;
    const bf16_t* q_scale; const bf16_t* k_scale;
    const float* pe;
    int64_t pe_batch_stride;
    int qk_cols, qk_heads, qk_seq_len, qk_out_len, qk_pos0;
    float qk_eps;
};

// One or two products of the same N and K (and the same epilogue form) that share a launch.
struct GemmSet {
    GemmParams p[2];
    int n;
};

// The two products of `args` as one launch of row vectors (M <= 8) beside other work: true where they can share one, and then g
// holds them. (product[1].M == 0: there is one product.) rc: what the arguments themselves come to.
bool rows_beside(const flux_linear_pair_args* args, GemmSet& g, int& rc);

}  // namespace flux
