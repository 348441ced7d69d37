// Row vectors (M <= 8) times a weight matrix, for launches of their own and beside other work.
#pragma once

#include "gemm_params.h"

namespace flux {

constexpr int kGemvCols = 2;  // output columns per wave

// The wave's columns from n0 on: bias, GELU, gated residual, each rounded like the tiled kernels' epilogue; lane 0 stores.
template <int MM>
__device__ __forceinline__ void gemv_store(const GemmParams& p, int n0, int lane, const float (&acc)[kGemvCols][MM], const bf16_t (&bias_raw)[kGemvCols]) {
    constexpr int CPW = kGemvCols;
    if (lane == 0) {
#pragma unroll
        for (int c = 0; c < CPW; ++c) {
            const int n = n0 + c;
            if (n >= p.N) break;
            const float b = bf2f(bias_raw[c]);
#pragma unroll
            for (int m = 0; m < MM; ++m) {
                float t = acc[c][m] + b;
                if (p.act == FLUX_ACT_GELU_TANH && n >= p.act_begin) t = gelu_tanh_f32(t);
                t = round_bf16(t);
                if (p.gate != nullptr) {
                    const float g = bf2f(p.gate[static_cast<int64_t>(m / p.rows_per_batch) * p.gate_stride + n]);
                    const float r = bf2f(p.resid[static_cast<int64_t>(m) * p.ldresid + n]);
                    t = r + round_bf16(g * t);
                }
                bf16_t* dst = n < p.split_n ? p.Y + static_cast<int64_t>(m) * p.ldy + n
                                            : p.Y2 + static_cast<int64_t>(m) * p.ldy2 + (n - p.split_n + p.y2_col0);
                *dst = f2bf(t);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Skinny problems (M <= 8, e.g. the Modulation projection of one conditioning vector per batch
// element): HBM-bound on W. A wave streams the W rows of two output columns with 16-byte loads,
// six or twelve in flight per lane, while the few activation rows come from cache; the dot products are
// folded with a wave butterfly. The kernel is instantiated per row count, so it has no row tests.
// Everything a wave needs beside W is requested in front of it: with the activation rows behind the W loads, and the
// bias behind the sums, each was a wait of its own while all waves of the launch stood at the same place. W is read
// once, so its loads mostly carry the non-temporal hint (a bare read of 113 MB: 18.4 -> 17.4 us). us, weights from HBM,
// before -> now: 1 x 9216 x 3072 with SiLU 14.0 -> 11.2 (the bare read 9.5), two such products of 18432 columns in one launch
// 38.7 -> 33.8 (6.7 TB/s), 3 rows 17.9 -> 15.8, 8 rows 33.6 -> 31.2, 1 x 3072 x 12288 22.3 -> 21.4.
// ------------------------------------------------------------------------------------------------
constexpr int kGemvSiluLds = 48 * 1024;  // bytes of LDS for the (activated) input rows (bf16)

// SILU_LDS: the few activation rows are staged in LDS once per workgroup, with the input activation
// x * sigmoid(x) applied on the way (rounded to bf16, as the separate operator would leave it). Every
// wave needs all K values of every row: read from memory inside the K loop they queue behind the W
// loads of the wave (the memory counter is in-order), and the activation, two transcendentals per
// value, would be repeated by each of the N / 2 waves. For the same reason the workgroup's share of them is
// requested in front of the first W loads, not behind. Rows that do not fit the LDS budget are read
// from memory as they are needed.
// U: 16-byte vectors of a W row a lane requests at once (see launch_gemv).
// EXACT: K = 512 * U, so every lane has exactly U vectors per row and the K loop runs once, without tests.
// ONCE: W is read with the non-temporal hint (see launch_gemv).
// block: which 4 * kGemvCols columns; act_lds: MM * K * 2 bytes with SILU_LDS.
template <int MM, bool SILU_LDS, int U, bool EXACT, bool ONCE>
__device__ __forceinline__ void gemv_small_m(const GemmParams& p, int block, char* act_lds) {
    constexpr int CPW = kGemvCols;  // CPW * U 16-byte loads of W in flight per lane
    // Activation vectors a thread requests in front: its share at K = 3072 where a whole such row of W is in flight, one or
    // two where half of it is (four rows of K = 1536: 5.4 us, 5.6 with two, 6.2 with all six).
    constexpr int PRE = U == 6 ? MM + (MM + 1) / 2 : (MM <= 4 ? 1 : 2);
    const int lane = threadIdx.x & 63;
    const int n0 = (block * 4 + (threadIdx.x >> 6)) * CPW;
    const bf16_t* wrow[CPW];
#pragma unroll
    for (int c = 0; c < CPW; ++c) wrow[c] = p.W + static_cast<int64_t>(n0 + c < p.N ? n0 + c : (n0 < p.N ? n0 : p.N - 1)) * p.ldw;
    const int act_n = MM * p.K;
    auto act_at = [&](int i) {   // K is a multiple of 8: a vector stays inside one row
        const int m = MM == 1 ? 0 : i / p.K, k = i - m * p.K;
        return p.A + static_cast<int64_t>(m) * p.lda + k;
    };
    // (the bias goes in front too: behind the sums it was a round trip to memory with nothing beside it)
    bf16_t bias_raw[CPW];
#pragma unroll
    for (int c = 0; c < CPW; ++c) bias_raw[c] = p.bias ? p.bias[min(n0 + c, p.N - 1)] : static_cast<bf16_t>(0);
    Vec16<bf16_t> pre[PRE];
    if (SILU_LDS) {
#pragma unroll
        for (int j = 0; j < PRE; ++j) {
            const int i = static_cast<int>(threadIdx.x) * 8 + j * 2048;
            pre[j] = ld16(act_at(i < act_n ? i : 0));
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // the first group of W loads goes out before the activation is worked on
    Vec16<bf16_t> w[U][CPW];
    auto request_w = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512;
            // past the end: a harmless re-read, skipped below
#pragma unroll
            for (int c = 0; c < CPW; ++c) {
                const bf16_t* const at = wrow[c] + (EXACT || k < p.K ? k : k0);
                w[u][c] = ONCE ? ld16_once(at) : ld16(at);
            }
        }
    };
    if (EXACT || lane * 8 < p.K) request_w(lane * 8);
    if (SILU_LDS) {
        __builtin_amdgcn_sched_barrier(0);
        bf16_t* dst = reinterpret_cast<bf16_t*>(act_lds);
        auto stage = [&](int i, const Vec16<bf16_t>& a) {
            Vec16<bf16_t> o = a;
            if (p.in_silu) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float f = bf2f(a.v[e]);
                    o.v[e] = f2bf(f * __builtin_amdgcn_rcpf(1.0f + __expf(-f)));
                }
            }
            *reinterpret_cast<Vec16<bf16_t>*>(dst + i) = o;
        };
#pragma unroll
        for (int j = 0; j < PRE; ++j) {
            const int i = static_cast<int>(threadIdx.x) * 8 + j * 2048;
            if (i < act_n) stage(i, pre[j]);
        }
        for (int i = threadIdx.x * 8 + PRE * 2048; i < act_n; i += 2048) stage(i, ld16(act_at(i)));
        __syncthreads();
    }
    if (n0 >= p.N) return;  // whole wave leaves together (after the barrier)
    float acc[CPW][MM];
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int m = 0; m < MM; ++m) acc[c][m] = 0.0f;
    for (int k0 = lane * 8; k0 < (EXACT ? 512 : p.K); k0 += 512 * U) {
        if (!EXACT && k0 != lane * 8) request_w(k0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512;
            if (!EXACT && k >= p.K) break;
            float af[MM][8];
#pragma unroll
            for (int m = 0; m < MM; ++m) {
                Vec16<bf16_t> a;
                if (SILU_LDS) a = *reinterpret_cast<const Vec16<bf16_t>*>(act_lds + (static_cast<size_t>(m) * p.K + k) * 2);
                else a = ld16(p.A + static_cast<int64_t>(m) * p.lda + k);
#pragma unroll
                for (int e = 0; e < 8; ++e) af[m][e] = bf2f(a.v[e]);
                if (!SILU_LDS && p.in_silu) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) af[m][e] = round_bf16(af[m][e] * __builtin_amdgcn_rcpf(1.0f + __expf(-af[m][e])));
                }
            }
#pragma unroll
            for (int c = 0; c < CPW; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float wf = bf2f(w[u][c].v[e]);
#pragma unroll
                    for (int m = 0; m < MM; ++m) acc[c][m] += wf * af[m][e];
                }
        }
    }
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int m = 0; m < MM; ++m) acc[c][m] = group_sum<64>(acc[c][m]);
    gemv_store<MM>(p, n0, lane, acc, bias_raw);
}

// The same for `groups` groups of columns from `first` on, for workgroups beside those of other work: these are few to a CU and
// have to keep W coming by themselves, so a wave requests the next half row or row of its two columns before it multiplies
// the last one. The activation rows are staged once.
// EXACT: K is a multiple of 512 * U.
template <int MM, int U, bool EXACT>
__device__ __forceinline__ void gemv_groups(const GemmParams& p, int first, int groups, char* act_lds) {
    constexpr int CPW = kGemvCols;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int act_n = MM * p.K, steps = (p.K + 512 * U - 1) / (512 * U);
    Vec16<bf16_t> w[2][U][CPW];
    bf16_t bias[2][CPW];
    // step `at` of the wave's sequence: U vectors a lane of its two columns; past the end of a row or of W, a harmless re-read
    auto column = [&](int at) { return (first + at / steps) * 4 * CPW + wave * CPW; };
    auto request = [&](int at, Vec16<bf16_t> (&to)[U][CPW], bf16_t (&b)[CPW]) {
        const int n0 = column(at), k0 = at % steps * (512 * U) + lane * 8;
#pragma unroll
        for (int c = 0; c < CPW; ++c) {
            const int n = min(n0 + c, p.N - 1);
            const bf16_t* const row = p.W + static_cast<int64_t>(n) * p.ldw;
            b[c] = p.bias ? p.bias[n] : static_cast<bf16_t>(0);
#pragma unroll
            for (int u = 0; u < U; ++u) to[u][c] = ld16_once(row + (EXACT || k0 + u * 512 < p.K ? k0 + u * 512 : 0));
        }
    };
    const int total = groups * steps;
    request(0, w[0], bias[0]);
    for (int i = threadIdx.x * 8; i < act_n; i += 2048) {
        const int m = MM == 1 ? 0 : i / p.K;
        Vec16<bf16_t> a = ld16(p.A + static_cast<int64_t>(m) * p.lda + (i - m * p.K));
        if (p.in_silu) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = bf2f(a.v[e]);
                a.v[e] = f2bf(f * __builtin_amdgcn_rcpf(1.0f + __expf(-f)));
            }
        }
        *reinterpret_cast<Vec16<bf16_t>*>(act_lds + i * 2) = a;
    }
    __syncthreads();
    float acc[CPW][MM];
    auto step = [&](int at, Vec16<bf16_t> (&from)[U][CPW], bf16_t (&b)[CPW]) {
        const int part = at % steps, k0 = part * (512 * U) + lane * 8;
        if (part == 0)
#pragma unroll
            for (int c = 0; c < CPW; ++c)
#pragma unroll
                for (int m = 0; m < MM; ++m) acc[c][m] = 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 512;
            if (!EXACT && k >= p.K) break;
#pragma unroll
            for (int m = 0; m < MM; ++m) {
                const Vec16<bf16_t> a = *reinterpret_cast<const Vec16<bf16_t>*>(act_lds + (static_cast<size_t>(m) * p.K + k) * 2);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float af = bf2f(a.v[e]);
#pragma unroll
                    for (int c = 0; c < CPW; ++c) acc[c][m] += bf2f(from[u][c].v[e]) * af;
                }
            }
        }
        if (part < steps - 1) return;
#pragma unroll
        for (int c = 0; c < CPW; ++c)
#pragma unroll
            for (int m = 0; m < MM; ++m) acc[c][m] = group_sum<64>(acc[c][m]);
        gemv_store<MM>(p, column(at), lane, acc, b);
    };
    for (int at = 0; at < total; at += 2) {
        if (at + 1 < total) request(at + 1, w[1], bias[1]);
        step(at, w[0], bias[0]);
        if (at + 1 >= total) break;
        if (at + 2 < total) request(at + 2, w[0], bias[0]);
        step(at + 1, w[1], bias[1]);
    }
}

}  // namespace flux
