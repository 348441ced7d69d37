// Row-wise, HBM-bound kernels: RMSNorm (fwd/bwd) and LayerNorm + adaLN modulation.
//
// Layout idea: a row is owned by a group of G adjacent lanes (G = 16, 32 or 64) and lives entirely
// in registers as ITER 16-byte vectors per lane, so each element crosses HBM exactly once in each
// direction and the reduction is a DPP butterfly with no LDS traffic. Rows too long for that
// (more than 64*ITER_MAX vectors) or not 16-byte addressable take a block-per-row kernel that
// re-reads the row from cache.
#include "common.h"
#include <algorithm>

namespace flux {

constexpr int kBlock = 256;

// ------------------------------------------------------------------------------------------------
// Register-resident row helpers
// ------------------------------------------------------------------------------------------------
template <typename T, int G, int ITER>
struct RowRegs {
    static constexpr int VEC = Elem<T>::VEC;
    float x[ITER][VEC];

    // col(it, lane) = (it*G + lane) * VEC
    __device__ __forceinline__ void load(const T* row, int lane, int n, bool row_ok) {
#pragma unroll
        for (int it = 0; it < ITER; ++it) {
            int c = (it * G + lane) * VEC;
            if (row_ok && c < n) {
                Vec16<T> v = ld16(row + c);
#pragma unroll
                for (int e = 0; e < VEC; ++e) x[it][e] = Elem<T>::load(v.v[e]);
            } else {
#pragma unroll
                for (int e = 0; e < VEC; ++e) x[it][e] = 0.0f;
            }
        }
    }
};

template <typename TS, int VEC>
__device__ __forceinline__ void load_vecf(const TS* p, float (&out)[VEC]) {
    // VEC consecutive elements of a small parameter vector (scale / shift), any alignment >= VEC*sizeof
    if constexpr (sizeof(TS) * VEC == 16) {
        Vec16<TS> v = ld16(p);
#pragma unroll
        for (int e = 0; e < VEC; ++e) out[e] = Elem<TS>::load(v.v[e]);
    } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) out[e] = Elem<TS>::load(p[e]);
    }
}

// ------------------------------------------------------------------------------------------------
// RMSNorm forward, register-resident.
// ------------------------------------------------------------------------------------------------
// R rows per thread (a block covers R * kBlock / G rows, row j of a thread being kBlock / G rows behind row
// j - 1). One row per thread is what is launched: two rows of one vector each, which put twice the loads
// in flight per wave and halve the number of workgroups, measured 14.7 us against 13.8 us at the Flux shape.
//
// One or two tensors of the same width and types per launch (t[1]'s blocks follow the blocks0 of t[0]): q and
// k of a q/k norm. At [1, 24, 256, 128] the kernel is 3 us of work behind a launch, and the second launch
// costs the host more than both kernels take.
template <typename T, typename TS>
struct RmsFwd {
    const T* x; const TS* scale; T* y; float* rstd;
    int64_t rows, d1, d2, s0, s1, s2;
};
template <typename T, typename TS>
struct RmsFwdSet {
    RmsFwd<T, TS> t[2];
    unsigned blocks0;
    int n;
    float eps;
};
template <typename T, typename TS, int G, int ITER, int R>
__global__ __launch_bounds__(kBlock) void rms_norm_fwd_regs(RmsFwdSet<T, TS> set) {
    const bool second = blockIdx.x >= set.blocks0;
    const RmsFwd<T, TS>& t = set.t[second];
    const unsigned block = blockIdx.x - (second ? set.blocks0 : 0u);
    const T* __restrict__ const x = t.x;
    const TS* __restrict__ const scale = t.scale;
    T* __restrict__ const y = t.y;
    float* __restrict__ const rstd_out = t.rstd;
    const int64_t rows = t.rows, d1 = t.d1, d2 = t.d2, s0 = t.s0, s1 = t.s1, s2 = t.s2;
    const int n = set.n;
    const float eps = set.eps;
    constexpr int VEC = Elem<T>::VEC;
    constexpr int ROWS_PER_PASS = kBlock / G;
    const int lane = threadIdx.x % G;
    const int64_t row0 = static_cast<int64_t>(block) * (ROWS_PER_PASS * R) + threadIdx.x / G;

    // Offset of a row in the strided [d0, d1, d2] view. The host merges dimensions whose strides
    // allow it, so an evenly strided tensor arrives as d1 = 1 and needs no division; other views
    // divide in 32 bits when the row count allows (a 64-bit division costs a hundred instructions,
    // which at one vector per lane is more than the rest of the kernel).
    auto offset_of = [&](int64_t row) -> int64_t {
        if (d1 == 1 && row < d2) return row * s2;
        if (rows <= 0x7fffffffLL) {
            const uint32_t r32 = static_cast<uint32_t>(row), e2 = static_cast<uint32_t>(d2), e1 = static_cast<uint32_t>(d1);
            const uint32_t t = r32 / e2, i2 = r32 - t * e2, i0 = t / e1, i1 = t - i0 * e1;
            return i0 * s0 + i1 * s1 + static_cast<int64_t>(i2) * s2;
        }
        const int64_t i2 = row % d2, t = row / d2;
        return (t / d1) * s0 + (t % d1) * s1 + i2 * s2;
    };
    RowRegs<T, G, ITER> r[R];
    bool row_ok[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int64_t row = row0 + j * ROWS_PER_PASS;
        row_ok[j] = row < rows;
        r[j].load(x + (row_ok[j] ? offset_of(row) : 0), lane, n, row_ok[j]);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int64_t row = row0 + j * ROWS_PER_PASS;
        float ss = 0.0f;
#pragma unroll
        for (int it = 0; it < ITER; ++it)
#pragma unroll
            for (int e = 0; e < VEC; ++e) ss += r[j].x[it][e] * r[j].x[it][e];
        ss = group_sum<G>(ss);
        const float rstd = rsqrtf(ss / static_cast<float>(n) + eps);

        if (!row_ok[j]) continue;
        if (rstd_out != nullptr && lane == 0) rstd_out[row] = rstd;
        T* yrow = y + row * n;
#pragma unroll
        for (int it = 0; it < ITER; ++it) {
            int c = (it * G + lane) * VEC;
            if (c < n) {
                float w[VEC];
                load_vecf<TS, VEC>(scale + c, w);
                Vec16<T> o;
#pragma unroll
                for (int e = 0; e < VEC; ++e) o.v[e] = Elem<T>::store(Elem<T>::round(r[j].x[it][e] * rstd) * w[e]);
                st16(yrow + c, o);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Block-wide sum for the block-per-row kernels.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ float block_sum(float v, float* lds /* >= 4 floats + 1 */) {
    v = group_sum<64>(v);
    const int wave = threadIdx.x / 64;
    __syncthreads();
    if (threadIdx.x % 64 == 0) lds[wave] = v;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) t += lds[w];
    return t;
}

// RMSNorm forward, one block per row, any n and alignment (VEC = 1) or 16-byte rows (VEC = Elem::VEC).
template <typename T, typename TS, int VEC>
__global__ __launch_bounds__(kBlock) void rms_norm_fwd_block(
    const T* __restrict__ x, const TS* __restrict__ scale, T* __restrict__ y, float* __restrict__ rstd_out,
    int64_t rows, int64_t d1, int64_t d2, int n, int64_t s0, int64_t s1, int64_t s2, float eps) {
    __shared__ float lds[8];
    const int64_t row = blockIdx.x;
    int64_t i2 = row % d2;
    int64_t t = row / d2;
    int64_t i1 = t % d1;
    int64_t i0 = t / d1;
    const T* xrow = x + i0 * s0 + i1 * s1 + i2 * s2;
    T* yrow = y + row * n;

    float ss = 0.0f;
    for (int c = threadIdx.x * VEC; c < n; c += kBlock * VEC) {
        if constexpr (VEC == 1) {
            float v = Elem<T>::load(xrow[c]);
            ss += v * v;
        } else {
            Vec16<T> v = ld16(xrow + c);
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                float f = Elem<T>::load(v.v[e]);
                ss += f * f;
            }
        }
    }
    ss = block_sum(ss, lds);
    const float rstd = rsqrtf(ss / static_cast<float>(n) + eps);
    if (rstd_out != nullptr && threadIdx.x == 0) rstd_out[row] = rstd;
    for (int c = threadIdx.x * VEC; c < n; c += kBlock * VEC) {
        if constexpr (VEC == 1) {
            float v = Elem<T>::load(xrow[c]);
            yrow[c] = Elem<T>::store(Elem<T>::round(v * rstd) * Elem<TS>::load(scale[c]));
        } else {
            Vec16<T> v = ld16(xrow + c);
            float w[VEC];
            load_vecf<TS, VEC>(scale + c, w);
            Vec16<T> o;
#pragma unroll
            for (int e = 0; e < VEC; ++e) o.v[e] = Elem<T>::store(Elem<T>::round(Elem<T>::load(v.v[e]) * rstd) * w[e]);
            st16(yrow + c, o);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// RMSNorm backward: dx = rstd*(dy*w) - rstd^3/n * sum(dy*w*x) * x ;  dscale += sum_rows dy*x*rstd.
// One group of G lanes per row (register-resident); each block reduces its rows' dscale partials in
// registers while its groups walk the block's rows, folds them in LDS and writes them as one row of
// `part` [blocks, n], which rms_norm_dscale_reduce adds up in a fixed order. Without a workspace
// (part = null) it finishes with one atomic per column per block into a dscale that the caller cleared.
// Bound by HBM: x and dy in, dx out. With the workspace [98304, 128] bf16 takes 22.4 us for both launches
// (75 MB, 3.4 TB/s) and [6144, 128] 7.0 us; clearing dscale, atomics and converting it took 27.2 and
// 14.1 us. Short rows (one vector per lane) run as 256 blocks of 1024 threads: 512 and 1024 blocks of 1024, 512
// or 256 threads take 22.8 to 25.1 us at the first shape and 7.1 to 7.4 us at the second, because the
// reduction reads a row of partials per block.
constexpr int kBwdThreads1 = 1024, kBwdBlocks1 = 256;

// ------------------------------------------------------------------------------------------------
template <typename T, typename TS, int G, int ITER, int BLK>
__global__ __launch_bounds__(BLK) void rms_norm_bwd_regs(
    const T* __restrict__ dy, const T* __restrict__ x, const TS* __restrict__ scale, const float* __restrict__ rstd_in,
    T* __restrict__ dx, float* __restrict__ dscale, float* __restrict__ part, int64_t rows, int n, int rows_per_group) {
    constexpr int VEC = Elem<T>::VEC;
    constexpr int GROUPS = BLK / G;
    const int lane = threadIdx.x % G;
    const int grp = threadIdx.x / G;

    float w[ITER][VEC];
    float dw[ITER][VEC];
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        int c = (it * G + lane) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) { w[it][e] = 0.0f; dw[it][e] = 0.0f; }
        if (c < n) load_vecf<TS, VEC>(scale + c, w[it]);
    }

    // A block owns GROUPS * rows_per_group consecutive rows and its groups take them interleaved, so
    // one step of the block reads a contiguous span; U rows per group are requested before the first
    // is used.
    constexpr int U = ITER == 1 ? 4 : (ITER == 2 ? 2 : 1);
    const int64_t block_row0 = static_cast<int64_t>(blockIdx.x) * GROUPS * rows_per_group;
    for (int i0 = 0; i0 < rows_per_group; i0 += U) {
        RowRegs<T, G, ITER> rx[U], rdy[U];
        float rstd[U];
        bool ok[U];
        int64_t row[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            row[u] = block_row0 + static_cast<int64_t>(i0 + u) * GROUPS + grp;
            ok[u] = i0 + u < rows_per_group && row[u] < rows;  // uniform over the group
            const int64_t r = ok[u] ? row[u] : 0;
            rx[u].load(x + r * n, lane, n, ok[u]);
            rdy[u].load(dy + r * n, lane, n, ok[u]);
            rstd[u] = ok[u] ? rstd_in[r] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float dot = 0.0f;
#pragma unroll
            for (int it = 0; it < ITER; ++it)
#pragma unroll
                for (int e = 0; e < VEC; ++e) dot += rdy[u].x[it][e] * w[it][e] * rx[u].x[it][e];
            dot = group_sum<G>(dot);
            const float coef = -rstd[u] * rstd[u] * rstd[u] * dot / static_cast<float>(n);
            if (ok[u]) {
#pragma unroll
                for (int it = 0; it < ITER; ++it) {
                    int c = (it * G + lane) * VEC;
                    if (c < n) {
                        Vec16<T> o;
#pragma unroll
                        for (int e = 0; e < VEC; ++e) {
                            o.v[e] = Elem<T>::store(rstd[u] * rdy[u].x[it][e] * w[it][e] + coef * rx[u].x[it][e]);
                            dw[it][e] += rdy[u].x[it][e] * rx[u].x[it][e] * rstd[u];
                        }
                        st16(dx + row[u] * n + c, o);
                    }
                }
            }
        }
    }
    // Fold the block's GROUPS partial rows in LDS.
    extern __shared__ float dw_lds[];  // [GROUPS][G*ITER*VEC]
    constexpr int COLS = G * ITER * VEC;
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        int c = (it * G + lane) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) dw_lds[grp * COLS + c + e] = dw[it][e];
    }
    __syncthreads();
    for (int c = threadIdx.x; c < n; c += BLK) {
        float t = 0.0f;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) t += dw_lds[g * COLS + c];
        if (part) part[static_cast<int64_t>(blockIdx.x) * n + c] = t;
        else atomicAdd(dscale + c, t);
    }
}

// dscale[c] = the sum of part[0 .. parts)[c], rounded once to dscale's type. A workgroup takes 32 columns
// with 32 threads each; a thread adds every 32nd part, the 32 sums are folded in LDS in order, so the
// result does not depend on timing. At 256 parts of 128 columns (128 KB, out of the L2s) all eight loads of
// a thread are in flight at once.
constexpr int kDscaleCols = 32, kDscaleStrips = 32;
template <typename TD>
__global__ __launch_bounds__(kDscaleCols * kDscaleStrips) void rms_norm_dscale_reduce(
    const float* __restrict__ part, TD* __restrict__ dscale, int parts, int n) {
    __shared__ float sums[kDscaleStrips][kDscaleCols];
    const int col = threadIdx.x % kDscaleCols, strip = threadIdx.x / kDscaleCols;
    const int c = blockIdx.x * kDscaleCols + col;
    float t = 0.0f;
    if (c < n) {
#pragma unroll 8
        for (int i = strip; i < parts; i += kDscaleStrips) t += part[static_cast<int64_t>(i) * n + c];
    }
    sums[strip][col] = t;
    __syncthreads();
    if (strip == 0 && c < n) {
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < kDscaleStrips; ++i) total += sums[i][col];
        dscale[c] = Elem<TD>::store(total);
    }
}

__global__ __launch_bounds__(kBlock) void zero_floats(float* __restrict__ p, int n) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// Block-per-row backward for rows that do not fit the register path.
template <typename T, typename TS>
__global__ __launch_bounds__(kBlock) void rms_norm_bwd_block(
    const T* __restrict__ dy, const T* __restrict__ x, const TS* __restrict__ scale, const float* __restrict__ rstd_in,
    T* __restrict__ dx, float* __restrict__ dscale, int64_t rows, int n) {
    __shared__ float lds[8];
    const int64_t row = blockIdx.x;
    const T* xr = x + row * n;
    const T* dyr = dy + row * n;
    const float rstd = rstd_in[row];
    float dot = 0.0f;
    for (int c = threadIdx.x; c < n; c += kBlock)
        dot += Elem<T>::load(dyr[c]) * Elem<TS>::load(scale[c]) * Elem<T>::load(xr[c]);
    dot = block_sum(dot, lds);
    const float coef = -rstd * rstd * rstd * dot / static_cast<float>(n);
    for (int c = threadIdx.x; c < n; c += kBlock) {
        float g = Elem<T>::load(dyr[c]), xv = Elem<T>::load(xr[c]);
        dx[row * n + c] = Elem<T>::store(rstd * g * Elem<TS>::load(scale[c]) + coef * xv);
        atomicAdd(dscale + c, g * xv * rstd);
    }
}

// ------------------------------------------------------------------------------------------------
// LayerNorm + modulation, register-resident: two-pass statistics on the registers.
// For bf16 storage the normalised value, (1+scale) and the product are each rounded to bf16 before
// the next step, the evaluation order of functional/normalization.py:6-12 on bf16 tensors.
// ------------------------------------------------------------------------------------------------
// One or two tensors of the same width per launch (t[1]'s blocks follow the blocks0 of t[0]): the text
// and the image rows of a double-stream block, whose text part is a few microseconds of work behind a
// launch of its own.
template <typename T>
struct LnMod {
    const T* x; const T* scale; const T* shift; T* y;
    int64_t rows, seq, mod_stride;
};
template <typename T>
struct LnModSet {
    LnMod<T> t[2];
    unsigned blocks0;
    int n;
    float eps;
    bool once;   // x is read past the caches (see ln_mod_launch)
};

// Straight-line: rows past the end and columns past n are clamped for the loads (x, scale and shift
// vectors all go out before the first reduction) and masked in the sums; only the stores are
// predicated. FULL = the row fills the lanes exactly (n == G * ITER * VEC), no column masks at all.
// MODLDS: all rows of a workgroup belong to one batch element, and the workgroup prepares that element's
// modulation vectors once, in LDS, as fp32: g = (1 + scale) rounded like the PyTorch op, and shift. Every
// row needs all of both vectors; loaded and converted by each wave for itself (MODLDS = false, the
// general form) that is as many loads as the row itself has and a fifth of the kernel's arithmetic.
template <typename T, int G, int ITER, bool FULL, bool MODLDS>
__global__ __launch_bounds__(kBlock) void ln_mod_fwd_regs(LnModSet<T> set) {
    const bool second = blockIdx.x >= set.blocks0;
    const LnMod<T>& t = set.t[second];
    const unsigned block = blockIdx.x - (second ? set.blocks0 : 0u);
    const T* __restrict__ const x = t.x;
    const T* __restrict__ const scale = t.scale;
    const T* __restrict__ const shift = t.shift;
    T* __restrict__ const y = t.y;
    const int64_t rows = t.rows, seq = t.seq, mod_stride = t.mod_stride;
    const int n = set.n;
    const float eps = set.eps;
    constexpr int VEC = Elem<T>::VEC;
    constexpr int ROWS_PER_BLOCK = kBlock / G;
    constexpr int NMAX = MODLDS ? G * ITER * VEC : 1;
    __shared__ __attribute__((aligned(16))) float g_lds[NMAX], d_lds[NMAX];
    const int lane = threadIdx.x % G;
    const int64_t row_raw = static_cast<int64_t>(block) * ROWS_PER_BLOCK + threadIdx.x / G;
    const bool row_ok = row_raw < rows;
    const int64_t row = row_ok ? row_raw : rows - 1;
    const int64_t b = row / seq;
    const T* xr = x + row * n;
    const T* sc = scale + b * mod_stride;
    const T* sh = shift + b * mod_stride;

    Vec16<T> xv[ITER], av[ITER], dv[ITER];
    bool in[ITER];
    const bool once = sizeof(T) == 4 && set.once;
#pragma unroll
    for (int it = 0; it < ITER; ++it) in[it] = FULL || (it * G + lane) * VEC < n;
    if (once) {
#pragma unroll
        for (int it = 0; it < ITER; ++it) xv[it] = ld16_once(xr + (in[it] ? (it * G + lane) * VEC : 0));
    } else {
#pragma unroll
        for (int it = 0; it < ITER; ++it) xv[it] = ld16(xr + (in[it] ? (it * G + lane) * VEC : 0));
    }
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int cl = in[it] ? (it * G + lane) * VEC : 0;
        if (!MODLDS) {
            av[it] = ld16(sc + cl);
            dv[it] = ld16(sh + cl);
        }
    }
    if (MODLDS) {
        // the first row's batch element is every row's (the host checks that a block does not span two)
        const int64_t b0 = (static_cast<int64_t>(block) * ROWS_PER_BLOCK) / seq;
        for (int c = threadIdx.x * VEC; c < n; c += kBlock * VEC) {
            const Vec16<T> a = ld16(scale + b0 * mod_stride + c), d = ld16(shift + b0 * mod_stride + c);
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                g_lds[c + e] = Elem<T>::round(1.0f + Elem<T>::load(a.v[e]));
                d_lds[c + e] = Elem<T>::load(d.v[e]);
            }
        }
    }
    float xf[ITER][VEC];
    float s = 0.0f;
#pragma unroll
    for (int it = 0; it < ITER; ++it)
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            xf[it][e] = in[it] ? Elem<T>::load(xv[it].v[e]) : 0.0f;
            s += xf[it][e];
        }
    s = group_sum<G>(s);
    const float mean = s / static_cast<float>(n);
    float q = 0.0f;
#pragma unroll
    for (int it = 0; it < ITER; ++it)
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float d = in[it] ? xf[it][e] - mean : 0.0f;
            q += d * d;
        }
    q = group_sum<G>(q);
    const float rstd = rsqrtf(q / static_cast<float>(n) + eps);
    if (MODLDS) __syncthreads();

    T* yrow = y + row * n;
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int c = (it * G + lane) * VEC;
        const int cl = in[it] ? c : 0;
        Vec16<T> o;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float nv = Elem<T>::round((xf[it][e] - mean) * rstd);
            const float g = MODLDS ? g_lds[cl + e] : Elem<T>::round(1.0f + Elem<T>::load(av[it].v[e]));
            const float d = MODLDS ? d_lds[cl + e] : Elem<T>::load(dv[it].v[e]);
            o.v[e] = Elem<T>::store(Elem<T>::round(nv * g) + d);
        }
        if (row_ok && in[it]) st16(yrow + c, o);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void ln_mod_fwd_block(
    const T* __restrict__ x, const T* __restrict__ scale, const T* __restrict__ shift, T* __restrict__ y,
    int64_t rows, int64_t seq, int n, int64_t mod_stride, float eps) {
    __shared__ float lds[8];
    const int64_t row = blockIdx.x;
    const T* xr = x + row * n;
    float s = 0.0f;
    for (int c = threadIdx.x; c < n; c += kBlock) s += Elem<T>::load(xr[c]);
    const float mean = block_sum(s, lds) / static_cast<float>(n);
    float q = 0.0f;
    for (int c = threadIdx.x; c < n; c += kBlock) {
        float d = Elem<T>::load(xr[c]) - mean;
        q += d * d;
    }
    const float rstd = rsqrtf(block_sum(q, lds) / static_cast<float>(n) + eps);
    const int64_t b = row / seq;
    const T* sc = scale + b * mod_stride;
    const T* sh = shift + b * mod_stride;
    for (int c = threadIdx.x; c < n; c += kBlock) {
        float nv = Elem<T>::round((Elem<T>::load(xr[c]) - mean) * rstd);
        float g = Elem<T>::round(1.0f + Elem<T>::load(sc[c]));
        y[row * n + c] = Elem<T>::store(Elem<T>::round(nv * g) + Elem<T>::load(sh[c]));
    }
}

// ------------------------------------------------------------------------------------------------
// Host dispatch
// ------------------------------------------------------------------------------------------------
struct RowPlan {
    int G;     // lanes per row, 0 = use the block kernel
    int ITER;  // vectors per lane
};

// Twelve vectors per lane is a float32 row of 3072 (48 registers of x). Left to the block-per-row kernel,
// which reads the row three times, element by element, layer norm + modulation of [4, 2048, 3072] fp32
// took 75 us (2.7 TB/s of the 201 MB it needs); held in registers it takes 41 us (4.9 TB/s; a 1 GiB copy
// on the same card 5.2 TB/s).
static RowPlan plan_row(int n, int vec) {
    if (n % vec != 0) return {0, 0};
    int nv = n / vec;
    if (nv <= 16) return {16, 1};
    if (nv <= 32) return {32, 1};
    if (nv <= 64) return {64, 1};
    int it = (nv + 63) / 64;
    const int allowed[] = {2, 3, 4, 6, 8, 12};
    for (int a : allowed)
        if (it <= a) return {64, a};
    return {0, 0};
}

#define FLUX_DISPATCH_GI(plan, CALL)                                   \
    do {                                                               \
        if (plan.G == 16) { CALL(16, 1); }                             \
        else if (plan.G == 32) { CALL(32, 1); }                        \
        else if (plan.ITER == 1) { CALL(64, 1); }                      \
        else if (plan.ITER == 2) { CALL(64, 2); }                      \
        else if (plan.ITER == 3) { CALL(64, 3); }                      \
        else if (plan.ITER == 4) { CALL(64, 4); }                      \
        else if (plan.ITER == 6) { CALL(64, 6); }                      \
        else if (plan.ITER == 8) { CALL(64, 8); }                      \
        else { CALL(64, 12); }                                         \
    } while (0)

// RMS norm reads a row twice in the block-per-row kernel, the second time from a cache, and needs many rows before a
// wave per row with twelve vectors per lane is the faster: us on the block kernel and in registers at 4608 bf16, 256 rows
// 3.8 and 5.8, 2048 rows 8.9 and 10.1, 3072 rows 13.5 and 12.8, 4096 rows 17.5 and 14.4; at 3072 fp32 3.8 and 4.8,
// 10.7 and 10.4, 17.6 and 13.7, 22.7 and 16.9.
constexpr int64_t kRmsLongRows = 2560;

template <typename T, typename TS>
static int rms_fwd_launch(const flux_rms_norm_args* a, int count, int n, float eps, hipStream_t st) {
    constexpr int VEC = Elem<T>::VEC;
    RowPlan plan = plan_row(n, VEC);
    int64_t most_rows = 0;
    for (int i = 0; i < count; ++i) most_rows = std::max(most_rows, a[i].d0 * a[i].d1 * a[i].d2);
    if (plan.ITER == 12 && most_rows < kRmsLongRows) plan = {0, 0};
    RmsFwdSet<T, TS> set;
    set.n = n;
    set.eps = eps;
    int used = 0;
    bool vec_ok[2];
    for (int i = 0; i < count; ++i) {
        int64_t d0 = a[i].d0, d1 = a[i].d1, d2 = a[i].d2, s0 = a[i].s0, s1 = a[i].s1, s2 = a[i].s2;
        const int64_t rows = d0 * d1 * d2;
        if (rows == 0) continue;
        vec_ok[used] = aligned16(a[i].x) && aligned16(a[i].y) && s0 % VEC == 0 && s1 % VEC == 0 && s2 % VEC == 0 &&
                       (sizeof(TS) * VEC != 16 || aligned16(a[i].scale));
        // merge dimensions that are evenly strided: [d0, d1, d2] -> [1, 1, rows] for a contiguous tensor
        if (d0 == 1 || s0 == d1 * s1) { d1 *= d0; d0 = 1; }
        if (d0 == 1 && (d1 == 1 || s1 == d2 * s2)) { d2 *= d1; d1 = 1; }
        set.t[used++] = {static_cast<const T*>(a[i].x), static_cast<const TS*>(a[i].scale), static_cast<T*>(a[i].y), a[i].rstd, rows, d1, d2, s0, s1, s2};
    }
    if (used == 0) return FLUX_OK;
    if (plan.G != 0 && vec_ok[0] && vec_ok[used - 1]) {
#define CALL(G_, I_)                                                                                          \
    do {                                                                                                      \
        constexpr int R_ = 1;   /* two short rows per thread measured 6 % slower at the Flux shape */            \
        constexpr int RPB_ = (kBlock / G_) * R_;                                                              \
        unsigned grid_ = 0;                                                                                   \
        for (int i = 0; i < used; ++i) {                                                                      \
            grid_ += (unsigned)((set.t[i].rows + RPB_ - 1) / RPB_);                                            \
            if (i == 0) set.blocks0 = grid_;                                                                  \
        }                                                                                                     \
        hipLaunchKernelGGL((rms_norm_fwd_regs<T, TS, G_, I_, R_>), dim3(grid_), dim3(kBlock), 0, st, set);     \
    } while (0)
        if (used == 1) set.t[1] = set.t[0];
        FLUX_DISPATCH_GI(plan, CALL);
#undef CALL
        return check_launch("flux_rms_norm");
    }
    for (int i = 0; i < used; ++i) {
        const RmsFwd<T, TS>& t = set.t[i];
        if (plan.G != 0 && vec_ok[i]) {   // the other one of a pair is not 16-byte addressable
            flux_rms_norm_args one = a[a[0].d0 * a[0].d1 * a[0].d2 == 0 ? 1 : i];
            const int rc = rms_fwd_launch<T, TS>(&one, 1, n, eps, st);
            if (rc != FLUX_OK) return rc;
        } else if (n % VEC == 0 && vec_ok[i]) {
            hipLaunchKernelGGL((rms_norm_fwd_block<T, TS, VEC>), dim3((unsigned)t.rows), dim3(kBlock), 0, st, t.x, t.scale, t.y, t.rstd,
                               t.rows, t.d1, t.d2, n, t.s0, t.s1, t.s2, eps);
        } else {
            hipLaunchKernelGGL((rms_norm_fwd_block<T, TS, 1>), dim3((unsigned)t.rows), dim3(kBlock), 0, st, t.x, t.scale, t.y, t.rstd,
                               t.rows, t.d1, t.d2, n, t.s0, t.s1, t.s2, eps);
        }
    }
    return check_launch("flux_rms_norm");
}

// How the register-resident backward splits `rows` rows; blocks == 0 where the row takes the block kernel.
struct BwdPlan {
    RowPlan row;
    int threads;         // per workgroup
    int rows_per_group;  // rows that a group of row.G lanes walks
    unsigned blocks;
};
static BwdPlan plan_bwd(int64_t rows, int n, int vec) {
    BwdPlan p = {plan_row(n, vec), 0, 0, 0};
    if (p.row.G == 0 || p.row.ITER > 4) return p;
    p.threads = p.row.ITER == 1 ? kBwdThreads1 : kBlock;
    const int64_t want = p.row.ITER == 1 ? kBwdBlocks1 : 1024, groups = p.threads / p.row.G;
    const int64_t rpg = (rows + want * groups - 1) / (want * groups);
    p.rows_per_group = static_cast<int>(rpg < 1 ? 1 : rpg);
    p.blocks = static_cast<unsigned>((rows + p.rows_per_group * groups - 1) / (p.rows_per_group * groups));
    return p;
}

template <typename TD>
static void dscale_reduce(const float* part, void* dscale, int parts, int n, hipStream_t st) {
    hipLaunchKernelGGL((rms_norm_dscale_reduce<TD>), dim3((n + kDscaleCols - 1) / kDscaleCols), dim3(kDscaleCols * kDscaleStrips), 0, st,
                       part, static_cast<TD*>(dscale), parts, n);
}

// With a workspace `ws` (plan_bwd's blocks * n floats, at least n) dscale is written, in dscale_dtype; without
// one it is fp32 and is added to.
template <typename T, typename TS>
static int rms_bwd_launch(const void* dy, const void* x, const void* scale, const float* rstd, void* dx, void* dscale, int dscale_dtype,
                          float* ws, int64_t rows, int n, hipStream_t st) {
    constexpr int VEC = Elem<T>::VEC;
    const T* dyp = static_cast<const T*>(dy);
    const T* xp = static_cast<const T*>(x);
    const TS* sp = static_cast<const TS*>(scale);
    T* dxp = static_cast<T*>(dx);
    const BwdPlan bp = plan_bwd(rows, n, VEC);
    const RowPlan plan = bp.row;
    const bool vec_ok = aligned16(dy) && aligned16(x) && aligned16(dx) && (sizeof(TS) * VEC != 16 || aligned16(scale));
    int parts = 0;
    if (rows > 0 && bp.blocks != 0 && vec_ok) {
#define CALL(G_, I_)                                                                                         \
    do {                                                                                                     \
        constexpr int IT = (I_ > 4 ? 4 : I_);                                                                \
        constexpr int BLK = IT == 1 ? kBwdThreads1 : kBlock;                                                 \
        const size_t lds_bytes = sizeof(float) * BLK * IT * VEC;                                             \
        hipLaunchKernelGGL((rms_norm_bwd_regs<T, TS, G_, IT, BLK>), dim3(bp.blocks), dim3(BLK), lds_bytes, st, dyp, xp, sp, \
                           rstd, dxp, static_cast<float*>(dscale), ws, rows, n, bp.rows_per_group);          \
    } while (0)
        FLUX_DISPATCH_GI(plan, CALL);
#undef CALL
        parts = static_cast<int>(bp.blocks);
    } else if (rows > 0) {   // sums by atomics: straight into an fp32 dscale
        float* const sums = ws && dscale_dtype == FLUX_BF16 ? ws : static_cast<float*>(dscale);
        if (ws) hipLaunchKernelGGL(zero_floats, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, sums, n);
        hipLaunchKernelGGL((rms_norm_bwd_block<T, TS>), dim3((unsigned)rows), dim3(kBlock), 0, st, dyp, xp, sp, rstd, dxp, sums, rows, n);
        if (sums == dscale) return check_launch("flux_rms_norm_bwd");
        parts = 1;
    }
    if (ws && dscale_dtype == FLUX_BF16) dscale_reduce<bf16_t>(ws, dscale, parts, n, st);
    else if (ws) dscale_reduce<float>(ws, dscale, parts, n, st);
    return check_launch("flux_rms_norm_bwd");
}

// fp32 inputs of more than a third of the 256 MiB cache in front of HBM are read with the non-temporal hint: what the
// operation in front read, the input that it wrote and this output do not fit there together. The hint favours programs
// whose tensors go through HBM. us, ordinary -> non-temporal, rows of 3072, six inputs and outputs in turn:
//                                             85.3 MiB       96 MiB         108 MiB        120 MiB          144 MiB
//   layer norm alone                        37.2 -> 32.6   41.5 -> 36.7   45.5 -> 40.6    48.7 -> 43.8    57.7 -> 52.8
//   behind an addition to other memory      79.7 -> 72.4   88.8 -> 83.2   99.8 -> 93.5   116.1 -> 104.9  136.9 -> 127.9
//   the same and a sum that reads y         93.6 -> 89.4  104.6 -> 100.7 119.0 -> 112.2  135.9 -> 123.8  158.4 -> 147.3
//   behind an addition in place             78.3 -> 73.7   87.3 -> 81.5   98.2 -> 91.5   110.9 -> 102.3  133.8 -> 122.9
// It costs where one input and one output take turns alone, which do fit: the same call again 30.1 -> 34.8 at 96 MiB, 37.3 -> 41.5 at
// 120, 45.3 -> 45.2 at 132; between two additions in place 87.5 -> 90.9, 108.1 -> 111.0, 124.0 -> 122.3. Smaller inputs mostly come
// from that cache (50 MB 15.5 -> 17.0), and bf16 gains a third of what fp32 does. (Stores with the hint make the call faster
// still, 10.3 us for 13.9 at [1, 4608, 3072] bf16, and the reader of the output slower: the single-stream block at 3 x 4336
// tokens 2840 -> 2873.)
constexpr int64_t kCacheBytes = 256 << 20;

template <typename T>
static int ln_mod_launch(const flux_layer_norm_args* a, int count, int n, float eps, hipStream_t st) {
    constexpr int VEC = Elem<T>::VEC;
    const RowPlan plan = plan_row(n, VEC);
    LnModSet<T> set;
    set.n = n;
    set.eps = eps;
    int used = 0;
    bool vec_ok = true;
    int64_t bytes = 0;
    for (int i = 0; i < count; ++i) {
        if (a[i].batch * a[i].seq == 0) continue;
        bytes += a[i].batch * a[i].seq * n * static_cast<int64_t>(sizeof(T));
        set.t[used++] = {static_cast<const T*>(a[i].x), static_cast<const T*>(a[i].scale), static_cast<const T*>(a[i].shift), static_cast<T*>(a[i].y),
                         a[i].batch * a[i].seq, a[i].seq, a[i].mod_batch_stride};
        vec_ok = vec_ok && aligned16(a[i].x) && aligned16(a[i].y) && aligned16(a[i].scale) && aligned16(a[i].shift) && a[i].mod_batch_stride % VEC == 0;
    }
    if (used == 0) return FLUX_OK;
    if (plan.G == 0 || !vec_ok) {
        for (int i = 0; i < used; ++i)
            hipLaunchKernelGGL((ln_mod_fwd_block<T>), dim3((unsigned)set.t[i].rows), dim3(kBlock), 0, st, set.t[i].x, set.t[i].scale, set.t[i].shift,
                               set.t[i].y, set.t[i].rows, set.t[i].seq, n, set.t[i].mod_stride, eps);
        return check_launch("flux_layer_norm_modulation");
    }
    if (used == 1) set.t[1] = set.t[0];
    set.once = 3 * bytes > kCacheBytes;
#define CALL(G_, I_)                                                                                        \
    do {                                                                                                    \
        constexpr int RPB_ = kBlock / G_;                                                                    \
        /* wave-per-row plans whose blocks stay inside one batch element stage the modulation vectors in LDS */ \
        bool lds_ = G_ == 64;                                                                               \
        unsigned grid_ = 0;                                                                                 \
        for (int i = 0; i < used; ++i) {                                                                    \
            lds_ = lds_ && (set.t[i].rows == set.t[i].seq || set.t[i].seq % RPB_ == 0);                      \
            grid_ += (unsigned)((set.t[i].rows + RPB_ - 1) / RPB_);                                          \
            if (i == 0) set.blocks0 = grid_;                                                                \
        }                                                                                                   \
        if (n == G_ * I_ * VEC && lds_)                                                                     \
            hipLaunchKernelGGL((ln_mod_fwd_regs<T, G_, I_, true, G_ == 64>), dim3(grid_), dim3(kBlock), 0, st, set);  \
        else if (n == G_ * I_ * VEC)                                                                        \
            hipLaunchKernelGGL((ln_mod_fwd_regs<T, G_, I_, true, false>), dim3(grid_), dim3(kBlock), 0, st, set);     \
        else if (lds_)                                                                                      \
            hipLaunchKernelGGL((ln_mod_fwd_regs<T, G_, I_, false, G_ == 64>), dim3(grid_), dim3(kBlock), 0, st, set); \
        else                                                                                                \
            hipLaunchKernelGGL((ln_mod_fwd_regs<T, G_, I_, false, false>), dim3(grid_), dim3(kBlock), 0, st, set);    \
    } while (0)
    FLUX_DISPATCH_GI(plan, CALL);
#undef CALL
    return check_launch("flux_layer_norm_modulation");
}

}  // namespace flux

using namespace flux;

static int rms_fwd_checked(const flux_rms_norm_args* a, int count, int32_t n, int32_t x_dtype, int32_t scale_dtype, float eps, void* stream) {
    int64_t rows = 0;
    for (int i = 0; i < count; ++i) {
        if (!a[i].x || !a[i].scale || !a[i].y) return fail(FLUX_E_NULL, "flux_rms_norm: null pointer");
        if (a[i].d0 < 0 || a[i].d1 < 0 || a[i].d2 < 0 || n <= 0)
            return fail(FLUX_E_SHAPE, "flux_rms_norm: bad shape [%lld,%lld,%lld,%d]", (long long)a[i].d0, (long long)a[i].d1, (long long)a[i].d2, n);
        rows += a[i].d0 * a[i].d1 * a[i].d2;
    }
    if (n > FLUX_MAX_ROW) return fail(FLUX_E_TOO_WIDE, "flux_rms_norm: n = %d exceeds the maximum row length %d", n, FLUX_MAX_ROW);
    if (rows == 0) return FLUX_OK;
    if (rows > 0x7fffffffLL * 4) return fail(FLUX_E_SHAPE, "flux_rms_norm: too many rows");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (x_dtype == FLUX_BF16 && scale_dtype == FLUX_BF16) return rms_fwd_launch<bf16_t, bf16_t>(a, count, n, eps, st);
    if (x_dtype == FLUX_BF16 && scale_dtype == FLUX_F32) return rms_fwd_launch<bf16_t, float>(a, count, n, eps, st);
    if (x_dtype == FLUX_F32 && scale_dtype == FLUX_F32) return rms_fwd_launch<float, float>(a, count, n, eps, st);
    return fail(FLUX_E_DTYPE, "flux_rms_norm: unsupported dtype pair (%d,%d)", x_dtype, scale_dtype);
}

extern "C" int flux_rms_norm(const void* x, const void* scale, void* y, float* rstd, int64_t d0, int64_t d1, int64_t d2,
                             int32_t n, int64_t s0, int64_t s1, int64_t s2, int32_t x_dtype, int32_t scale_dtype,
                             float eps, void* stream) {
    const flux_rms_norm_args a = {x, scale, y, rstd, d0, d1, d2, s0, s1, s2};
    return rms_fwd_checked(&a, 1, n, x_dtype, scale_dtype, eps, stream);
}

extern "C" int flux_rms_norm_pair(const flux_rms_norm_args* first, const flux_rms_norm_args* second, int32_t n,
                                  int32_t x_dtype, int32_t scale_dtype, float eps, void* stream) {
    if (!first || !second) return fail(FLUX_E_NULL, "flux_rms_norm_pair: null args");
    const flux_rms_norm_args a[2] = {*first, *second};
    return rms_fwd_checked(a, 2, n, x_dtype, scale_dtype, eps, stream);
}

static int rms_bwd_checked(const void* dy, const void* x, const void* scale, const float* rstd, void* dx, void* dscale, int dscale_dtype,
                           float* ws, int64_t rows, int32_t n, int32_t x_dtype, int32_t scale_dtype, void* stream) {
    if (!dy || !x || !scale || !rstd || !dx || !dscale) return fail(FLUX_E_NULL, "flux_rms_norm_bwd: null pointer");
    if (rows < 0 || n <= 0) return fail(FLUX_E_SHAPE, "flux_rms_norm_bwd: bad shape [%lld,%d]", (long long)rows, n);
    if (n > FLUX_MAX_ROW) return fail(FLUX_E_TOO_WIDE, "flux_rms_norm_bwd: n = %d exceeds the maximum row length %d", n, FLUX_MAX_ROW);
    if (rows == 0 && !ws) return FLUX_OK;
    if (rows > 0x7fffffffLL) return fail(FLUX_E_SHAPE, "flux_rms_norm_bwd: too many rows");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (x_dtype == FLUX_BF16 && scale_dtype == FLUX_BF16) return rms_bwd_launch<bf16_t, bf16_t>(dy, x, scale, rstd, dx, dscale, dscale_dtype, ws, rows, n, st);
    if (x_dtype == FLUX_BF16 && scale_dtype == FLUX_F32) return rms_bwd_launch<bf16_t, float>(dy, x, scale, rstd, dx, dscale, dscale_dtype, ws, rows, n, st);
    if (x_dtype == FLUX_F32 && scale_dtype == FLUX_F32) return rms_bwd_launch<float, float>(dy, x, scale, rstd, dx, dscale, dscale_dtype, ws, rows, n, st);
    return fail(FLUX_E_DTYPE, "flux_rms_norm_bwd: unsupported dtype pair (%d,%d)", x_dtype, scale_dtype);
}

extern "C" int flux_rms_norm_bwd(const void* dy, const void* x, const void* scale, const float* rstd, void* dx,
                                 float* dscale, int64_t rows, int32_t n, int32_t x_dtype, int32_t scale_dtype,
                                 void* stream) {
    return rms_bwd_checked(dy, x, scale, rstd, dx, dscale, FLUX_F32, nullptr, rows, n, x_dtype, scale_dtype, stream);
}

extern "C" int64_t flux_rms_norm_bwd_workspace_bytes(int64_t rows, int32_t n, int32_t x_dtype) {
    if (rows < 0 || rows > 0x7fffffffLL || n <= 0 || n > FLUX_MAX_ROW) return 0;
    const int64_t blocks = plan_bwd(rows, n, x_dtype == FLUX_BF16 ? Elem<bf16_t>::VEC : Elem<float>::VEC).blocks;
    return static_cast<int64_t>(sizeof(float)) * n * (blocks > 1 ? blocks : 1);
}

extern "C" int flux_rms_norm_bwd_ws(const void* dy, const void* x, const void* scale, const float* rstd, void* dx,
                                    void* dscale, int32_t dscale_dtype, void* ws, int64_t ws_bytes, int64_t rows, int32_t n,
                                    int32_t x_dtype, int32_t scale_dtype, void* stream) {
    if (!ws) return fail(FLUX_E_NULL, "flux_rms_norm_bwd_ws: null workspace");
    if (dscale_dtype != FLUX_BF16 && dscale_dtype != FLUX_F32) return fail(FLUX_E_DTYPE, "flux_rms_norm_bwd_ws: unsupported dscale dtype %d", dscale_dtype);
    if (reinterpret_cast<uintptr_t>(ws) % sizeof(float) != 0) return fail(FLUX_E_ALIGN, "flux_rms_norm_bwd_ws: the workspace must be 4-byte aligned");
    if (ws_bytes < flux_rms_norm_bwd_workspace_bytes(rows, n, x_dtype)) return fail(FLUX_E_SHAPE, "flux_rms_norm_bwd_ws: workspace of %lld bytes is too small", (long long)ws_bytes);
    return rms_bwd_checked(dy, x, scale, rstd, dx, dscale, dscale_dtype, static_cast<float*>(ws), rows, n, x_dtype, scale_dtype, stream);
}

static int ln_mod_checked(const flux_layer_norm_args* a, int count, int32_t n, int32_t dtype, float eps, void* stream) {
    int64_t rows = 0;
    for (int i = 0; i < count; ++i) {
        if (!a[i].x || !a[i].scale || !a[i].shift || !a[i].y) return fail(FLUX_E_NULL, "flux_layer_norm_modulation: null pointer");
        if (a[i].batch < 0 || a[i].seq < 0 || n <= 0) return fail(FLUX_E_SHAPE, "flux_layer_norm_modulation: bad shape [%lld,%lld,%d]", (long long)a[i].batch, (long long)a[i].seq, n);
        rows += a[i].batch * a[i].seq;
    }
    if (n > FLUX_MAX_ROW) return fail(FLUX_E_TOO_WIDE, "flux_layer_norm_modulation: n = %d exceeds the maximum row length %d", n, FLUX_MAX_ROW);
    if (rows == 0) return FLUX_OK;
    if (rows > 0x7fffffffLL) return fail(FLUX_E_SHAPE, "flux_layer_norm_modulation: too many rows");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (dtype == FLUX_BF16) return ln_mod_launch<bf16_t>(a, count, n, eps, st);
    if (dtype == FLUX_F32) return ln_mod_launch<float>(a, count, n, eps, st);
    return fail(FLUX_E_DTYPE, "flux_layer_norm_modulation: unsupported dtype %d", dtype);
}

extern "C" int flux_layer_norm_modulation(const void* x, const void* scale, const void* shift, void* y, int64_t batch,
                                          int64_t seq, int32_t n, int64_t mod_batch_stride, int32_t dtype, float eps,
                                          void* stream) {
    const flux_layer_norm_args a = {x, scale, shift, y, batch, seq, mod_batch_stride};
    return ln_mod_checked(&a, 1, n, dtype, eps, stream);
}

extern "C" int flux_layer_norm_modulation_pair(const flux_layer_norm_args* first, const flux_layer_norm_args* second, int32_t n,
                                               int32_t dtype, float eps, void* stream) {
    if (!first || !second) return fail(FLUX_E_NULL, "flux_layer_norm_modulation_pair: null args");
    const flux_layer_norm_args a[2] = {*first, *second};
    return ln_mod_checked(a, 2, n, dtype, eps, stream);
}
