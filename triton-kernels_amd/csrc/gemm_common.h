// Shared by the tiled GEMM translation units (gemm_bf16.hip: large tiles, gemm_pair.hip: eight-wave tiles):
// parameters, tile order, LDS loads and the epilogues of the rectangular tiles.
#pragma once

#include "common.h"
#include "gemm_params.h"
#include <type_traits>

namespace flux {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// One launch of a tiled kernel over the tile grid of a set: the tile rows of the second product follow
// those of the first, so the tile orders below see one grid of tiles_m x tiles_n.
struct GemmLaunch {
    GemmParams p[2];
    int tiles_m, tiles_n, group_m;
    int tiles_m0;               // tile rows of the first product
    int splits;                 // > 1: every tile's K range is cut into this many parts, each a workgroup of its own
    int slabs_per_split;
    bool take_turns;            // eight-wave tiles: neighbours walk K in orders of their own (gemm_pair.hip)
    float* partial;             // splits > 1: fp32 accumulators, [splits][tiles][4 waves][fragments][64 lanes][4]
};

constexpr int kGemmThreads = 256;
constexpr int kGemmCUs = 256;      // compute units of the one device this library is built for
constexpr unsigned kRsrcFlags = 0x00020000u;  // raw buffer, 32-bit data format
// A byte offset no buffer of ours reaches (record counts stay below 2^31, and so does k*2 added to
// it): the buffer load returns zeros for it, which is how rows past M/N and the K tail are padded.
constexpr uint32_t kOutOfRange = 0x80000000u;

// LDS-direct buffer loads are counted by vmcnt; the workgroup barrier alone does not wait for them.

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// Two floats -> one dword of two bf16 (a in the low half): a single v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t pack2_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ u32x2 pack4_bf16(float a, float b, float c, float d) {
    u32x2 r;
    r.x = pack2_bf16(a, b);
    r.y = pack2_bf16(c, d);
    return r;
}

// XCD-aware tile order. Workgroups are handed to the 8 XCDs round-robin, so workgroup w runs on
// XCD w % 8; giving each XCD one contiguous range of the (grouped) tile sequence makes the ~32 tiles
// resident on an XCD at any time a compact group_m x (32/group_m) patch that shares A and W panels
// in that XCD's L2.
// Tile order of a launch with the q/k epilogue. Its q/k tiles cost more than the others, each XCD
// owns one contiguous range of the tile sequence and works through it alone, and in the natural
// order one XCD would get twice its share of q/k tiles and another none. Here the q/k columns and
// the other columns form two sequences (each grouped like the plain order, so that the tiles
// resident on an XCD still share panels, and the q/k tiles of a patch the same rows of the rotation
// table), and every XCD takes its eighth of the first followed by its eighth of the second.
__device__ __forceinline__ bool tile_of_block_qk(const GemmLaunch& L, int bn, int& tm, int& tn) {
    const int nq = L.p[0].qk_cols / bn;
    const int Q = L.tiles_m * nq, R = L.tiles_m * (L.tiles_n - nq);
    const int per_xcd = gridDim.x / 8;
    const int x = blockIdx.x % 8, i = blockIdx.x / 8;
    const int q0 = x * Q / 8, q1 = (x + 1) * Q / 8;
    int u, cols, col0;
    if (i < q1 - q0) {
        u = q0 + i; cols = nq; col0 = 0;
    } else {
        u = x * per_xcd - q0 + (i - (q1 - q0)); cols = L.tiles_n - nq; col0 = nq;
        if (u >= R) return false;
    }
    const int width = L.group_m * cols;
    const int first_m = (u / width) * L.group_m;
    const int gsz = min(L.tiles_m - first_m, L.group_m);
    const int in_group = u % width;
    tm = first_m + in_group % gsz;
    tn = col0 + in_group / gsz;
    return true;
}

__device__ __forceinline__ void tile_at(const GemmLaunch& L, int t, int& tm, int& tn) {
    const int width = L.group_m * L.tiles_n;
    const int first_m = (t / width) * L.group_m;
    const int gsz = min(L.tiles_m - first_m, L.group_m);
    const int in_group = t % width;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

__device__ __forceinline__ bool tile_of_block(const GemmLaunch& L, int& tm, int& tn) {
    const int per_xcd = gridDim.x / 8;
    const int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (t >= L.tiles_m * L.tiles_n) return false;
    tile_at(L, t, tm, tn);
    return true;
}

// Which product tile row tm belongs to; tm becomes the row inside it. The kernels take that product's parameters
// as a copy: through a reference with an index that is not a constant, the compiler loads every field again at each
// use behind a store or a barrier, 719 scalar loads in the 256-wide tile's kernel, each with a wait for the LDS too.
// Fused q/k projection of the single block on that tile: 4608 rows 507 -> 499 us, 640 rows 94 -> 88 us.
__device__ __forceinline__ int product_of_tile(const GemmLaunch& L, int& tm) {
    const int second = tm >= L.tiles_m0 ? 1 : 0;
    tm -= second ? L.tiles_m0 : 0;
    return second;
}

// Element offset of row m of A.
__device__ __forceinline__ int64_t row_of_a(const GemmParams& p, int m) {
    int64_t o = m * p.lda;
    if (p.a_skip != 0) o += (static_cast<uint32_t>(m) / static_cast<uint32_t>(p.a_rows)) * p.a_skip;
    return o;
}

// One buffer load of 64 x 16 bytes, written by the memory pipeline straight into LDS at dst
// (+ lane * 16, implied by the instruction). `soff` is the scalar byte offset of the slab inside the
// rows; a vector offset with the top bit set is out of range for the resource and yields zeros.
__device__ __forceinline__ void load_chunk(__amdgpu_buffer_rsrc_t rsrc, char* dst, uint32_t voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}

__device__ __forceinline__ void wait_vmem_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Epilogue shared by the tiled kernels. A lane's accumulators hold one activation row and runs of
// 4 consecutive output columns. Per 32-row block: bias and GELU in fp32, one rounding to bf16, the
// block is parked in LDS (a private region per wave, overlaying the ring, which the caller's final
// barrier has retired) and leaves as 16-byte row segments, where the optional gated residual is
// applied. Interior tiles with 16-byte addressable outputs take a branch-free path; edge tiles and
// unaligned outputs take the checked path.
__device__ __forceinline__ float tanh_gelu_fast(float x) {
    // x * sigmoid(2u), u = sqrt(2/pi) (x + 0.044715 x^3), with log2(e) folded into the constants
    const float x2 = x * x;
    const float t = __builtin_fmaf(x2, -0.10294324f, -2.3022082f);
    const float e = __builtin_amdgcn_exp2f(x * t);
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// Epilogue for a wave whose 128 columns are one head of q or k: y = A W^T + bias is rounded to bf16
// (the projection's output), RMS-normalised over the head (x * rstd rounded, times scale rounded),
// rotated by the 2x2 matrices of its position and written to [B, heads, out_len, 128]. A lane holds
// 32 of a row's 128 columns; the other 96 are in the lanes 16, 32 and 48 further on, so the sum of
// squares takes two cross-lane steps. RAGGED = false: the tile is interior and lies inside one batch
// element, so its rows are consecutive positions of one (batch, head). RAGGED = true: the tile may run
// past the last row and may hold the last rows of one batch element followed by the first of the next
// (at most one such boundary: sequences are at least a tile long); rows past the end are computed on
// clamped table rows and not stored, rows behind the boundary take their table rows and their
// destination from the next batch element.
// FM fragment rows per wave in the tile, of which `acc` holds ROWS from `row0` on.
template <int FM, int NJ, int ROWS, bool RAGGED>
__device__ __forceinline__ void gemm_epilogue_qk(const GemmParams& p, f32x4 (&acc)[ROWS][2 * NJ], char* lds, int m0, int n0,
                                                 int row0, int wave, int lane) {
    constexpr int WROWS = 16 * ROWS, WCOLS = 32 * NJ;
    static_assert(WCOLS == 128, "a wave's columns are one head of 128");
    constexpr int C_PITCH = WCOLS * 2, C_CH = WCOLS / 8;
    constexpr int RPI = 64 / C_CH;
    constexpr int NIT = 16 / RPI;      // accesses per 16-row step
    constexpr int NQ = 2 * NJ;
    const int wm = wave >> 1, wn = wave & 1;
    const int frow = lane & 15, fq = lane >> 4;
    char* cw = lds + wave * (WROWS * C_PITCH);
    const int wave_n0 = n0 + wn * WCOLS;
    const int wave_m0 = m0 + wm * (16 * FM) + row0 * 16;
    const int hcol = wave_n0 / WCOLS;
    const bool is_k = hcol >= p.qk_heads;
    const int head = is_k ? hcol - p.qk_heads : hcol;
    const int batch = m0 / p.qk_seq_len;                        // the whole tile is in one batch element
    const int pos_w = p.qk_pos0 + (wave_m0 - batch * p.qk_seq_len);   // output row of the wave's first row

    // bias and scale of this lane's columns stay packed (two bf16 per register) and are unpacked at
    // their use: the epilogue needs its registers for the rotation entries in flight
    u32x2 bvp[NQ], scp[NQ];
    {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(is_k ? p.k_scale : p.q_scale), 0, WCOLS * 2, kRsrcFlags);
#pragma unroll
        for (int q = 0; q < NQ; ++q) scp[q] = __builtin_amdgcn_raw_buffer_load_b64(rs, (q * 16 + fq * 4) * 2, 0, 0);
    }
    if (p.bias != nullptr) {
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.bias), 0, p.N * 2, kRsrcFlags);
#pragma unroll
        for (int q = 0; q < NQ; ++q) bvp[q] = __builtin_amdgcn_raw_buffer_load_b64(rb, (wave_n0 + q * 16 + fq * 4) * 2, 0, 0);
    } else {
#pragma unroll
        for (int q = 0; q < NQ; ++q) bvp[q] = u32x2{0u, 0u};
    }
    auto unpack = [](u32x2 v, int e) -> float {
        const uint32_t w = e < 2 ? v.x : v.y;
        return __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
    };

    int waddr[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) waddr[q] = frow * C_PITCH + (((q * 2 + (fq >> 1)) ^ (frow & (C_CH - 1))) * 16) + (fq & 1) * 8;
    const int rrow = lane / C_CH, rch = lane % C_CH;
    int raddr[NIT];
#pragma unroll
    for (int t = 0; t < NIT; ++t) {
        const int row = t * RPI + rrow;
        raddr[t] = row * C_PITCH + ((rch ^ (row & (C_CH - 1))) * 16);
    }
    // rotation table of this lane's columns: 8 floats per quad, row stride 2 * 128 floats
    const float* pe_lane = p.pe + static_cast<int64_t>(batch) * p.pe_batch_stride + static_cast<int64_t>(pos_w + frow) * (2 * WCOLS) + fq * 8;
    // RAGGED: rows of the wave's sub-tile from `boundary` on belong to the next batch element, whose
    // positions restart: their table row is pe_next floats and their output row out_next bytes further on
    const int boundary = RAGGED ? (batch + 1) * p.qk_seq_len - wave_m0 : WROWS;
    const int64_t pe_next = RAGGED ? p.pe_batch_stride - static_cast<int64_t>(p.qk_seq_len) * (2 * WCOLS) : 0;
    const uint32_t out_next = RAGGED ? static_cast<uint32_t>((static_cast<int64_t>(p.qk_heads) * p.qk_out_len - p.qk_seq_len) * (WCOLS * 2)) : 0u;
    const int rows_valid = RAGGED ? p.M - wave_m0 : WROWS;   // rows of the sub-tile inside the matrix
    if (RAGGED && rows_valid <= 0) return;                   // nothing of this wave's to store (no workgroup barrier follows)
    char* dst_u = reinterpret_cast<char*>((is_k ? p.k_out : p.q_out) +
                                          ((static_cast<int64_t>(batch) * p.qk_heads + head) * p.qk_out_len + pos_w) * WCOLS);
    const uint32_t dst_lane = static_cast<uint32_t>(rrow * (WCOLS * 2) + rch * 16);
    const float inv_d = 1.0f / static_cast<float>(WCOLS);

#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        {
            // the step's rotation entries (from L2) are requested first and land while the sum of
            // squares is formed; the scheduling barrier keeps the compiler from sinking the loads
            // to their uses, where each would be waited for in turn
            f32x4 fr[NQ][2];
            {
                const float* pr = pe_lane + i * 16 * (2 * WCOLS);
                if (RAGGED) {
                    const int r = min(i * 16 + frow, rows_valid - 1);   // past the end: the last valid row's entries
                    pr = pe_lane + static_cast<int64_t>(r - frow) * (2 * WCOLS) + (r >= boundary ? pe_next : 0);
                }
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    fr[q][0] = *reinterpret_cast<const f32x4*>(pr + q * 32);
                    fr[q][1] = *reinterpret_cast<const f32x4*>(pr + q * 32 + 4);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // roundings to bf16 two values at a time: one v_cvt_pk_bf16_f32, then the halves widened again
            auto round2 = [](float a, float b, float& ra, float& rb) {
                const uint32_t w = pack2_bf16(a, b);
                ra = __uint_as_float(w << 16);
                rb = __uint_as_float(w & 0xffff0000u);
            };
            float x[NQ][4];
            float ss = 0.0f;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
#pragma unroll
                for (int e = 0; e < 4; e += 2)
                    round2(acc[i][q][e] + unpack(bvp[q], e), acc[i][q][e + 1] + unpack(bvp[q], e + 1), x[q][e], x[q][e + 1]);
#pragma unroll
                for (int e = 0; e < 4; ++e) ss += x[q][e] * x[q][e];
            }
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            const float rstd = rsqrtf(ss * inv_d + p.qk_eps);
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const f32x4 f0 = fr[q][0];
                const f32x4 f1 = fr[q][1];
                float xn[4];
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    float a, b;
                    round2(x[q][e] * rstd, x[q][e + 1] * rstd, a, b);
                    round2(a * unpack(scp[q], e), b * unpack(scp[q], e + 1), xn[e], xn[e + 1]);
                }
                const float o0 = f0[0] * xn[0] + f0[1] * xn[1];
                const float o1 = f0[2] * xn[0] + f0[3] * xn[1];
                const float o2 = f1[0] * xn[2] + f1[1] * xn[3];
                const float o3 = f1[2] * xn[2] + f1[3] * xn[3];
                *reinterpret_cast<u32x2*>(cw + i * 16 * C_PITCH + waddr[q]) = pack4_bf16(o0, o1, o2, o3);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int row_u = i * 16 + it * RPI;
            const Vec16<bf16_t> y = *reinterpret_cast<const Vec16<bf16_t>*>(cw + i * 16 * C_PITCH + raddr[it]);
            if (RAGGED) {
                const int r = row_u + rrow;
                if (r < rows_valid)
                    *reinterpret_cast<Vec16<bf16_t>*>(dst_u + static_cast<int64_t>(row_u) * (WCOLS * 2) + (dst_lane + (r >= boundary ? out_next : 0u))) = y;
            } else {
                *reinterpret_cast<Vec16<bf16_t>*>(dst_u + static_cast<int64_t>(row_u) * (WCOLS * 2) + dst_lane) = y;
            }
        }
    }
}

template <int K>
using ic = std::integral_constant<int, K>;

template <int N>
__device__ __forceinline__ void wait_loads_and_barrier() {
    // all but the newest N buffer loads of this wave have landed, its LDS reads have returned; the
    // memory clobber keeps LDS accesses on their side of the barrier
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Epilogue of the rectangular tile, for ROWS of the wave's FM fragment rows from `row0` on: per 16-row
// fragment row, bias (and GELU) in fp32, one rounding, the 16 x WCOLS block parked in LDS and read back as
// 16-byte row segments, lane l of access a taking segment a * 64 + l. A wave's columns are all on one
// side of split_n and of act_begin, and N is a multiple of 8 (the host checks). With a gate the residual
// rows are requested a fragment row ahead, the gate vectors once. EDGE: the tile may run past the last
// row or column, or hold rows of several batch elements: every row's gate vector is requested with its
// residual row.
// bytes of LDS: two fragment rows per wave
constexpr int rect_epilogue_lds(int fn) { return 4 * 2 * 16 * (16 * fn * 2 + 16); }
template <int FM, int FN, int ROWS, bool GELU, bool GATE, bool EDGE>
__device__ __forceinline__ void gemm_epilogue_rect(const GemmParams& p, f32x4 (&acc)[ROWS][FN], char* lds, int m0, int n0, int row0, int wave, int lane) {
    constexpr int WROWS = 16 * FM, WCOLS = 16 * FN;
    constexpr int C_CH = WCOLS / 8;               // 16-byte segments per row
    constexpr int C_PITCH = WCOLS * 2 + 16;       // padded: an odd number of 16-byte units spreads the rows over the banks
    constexpr int SEGS = 16 * C_CH;
    constexpr int NACC = (SEGS + 63) / 64;        // wave-wide accesses per fragment row
    const int wm = wave >> 1, wn = wave & 1;
    const int frow = lane & 15, fq = lane >> 4;
    char* cw = lds + wave * (2 * 16 * C_PITCH);   // two fragment rows per wave, used in turn
    const int wave_n0 = n0 + wn * WCOLS;
    const int wave_m0 = m0 + wm * WROWS + row0 * 16;
    const int rows_valid = EDGE ? p.M - wave_m0 : ROWS * 16;
    if (EDGE && (rows_valid <= 0 || wave_n0 >= p.N)) return;

    float bv[FN][4];
    if (p.bias != nullptr) {
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.bias), 0, p.N * 2, kRsrcFlags);
#pragma unroll
        for (int q = 0; q < FN; ++q) {
            const u32x2 raw = __builtin_amdgcn_raw_buffer_load_b64(rb, (wave_n0 + q * 16 + fq * 4) * 2, 0, 0);
            bv[q][0] = __uint_as_float(raw.x << 16);
            bv[q][1] = __uint_as_float(raw.x & 0xffff0000u);
            bv[q][2] = __uint_as_float(raw.y << 16);
            bv[q][3] = __uint_as_float(raw.y & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int q = 0; q < FN; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[q][e] = 0.0f;
    }
    const int waddr = frow * C_PITCH + fq * 8;    // + q * 32: column quad q of this lane's row
    const bool to_y = wave_n0 < p.split_n;
    const int64_t dst_ld = to_y ? p.ldy : p.ldy2;
    int raddr[NACC], srow[NACC];
    uint32_t dst_lane[NACC], res_lane[NACC];
    Vec16<bf16_t> gt[GATE && !EDGE ? NACC : 1];
#pragma unroll
    for (int a = 0; a < NACC; ++a) {
        // lanes past the last segment of a partial access take its place: their loads stay inside the 16 rows
        const int seg = SEGS % 64 == 0 ? a * 64 + lane : min(a * 64 + lane, SEGS - 1), row = seg / C_CH, ch = seg % C_CH;
        srow[a] = row;
        raddr[a] = row * C_PITCH + ch * 16;
        dst_lane[a] = static_cast<uint32_t>(row * dst_ld * 2 + ch * 16);
        res_lane[a] = 0;
        if (GATE && !EDGE) {
            gt[a] = ld16(p.gate + static_cast<int64_t>(m0 / p.rows_per_batch) * p.gate_stride + wave_n0 + ch * 8);
            res_lane[a] = static_cast<uint32_t>(row * p.ldresid * 2 + ch * 16);
        }
    }
    char* const dst_u = reinterpret_cast<char*>((to_y ? p.Y + wave_n0 : p.Y2 + (wave_n0 - p.split_n + p.y2_col0)) + static_cast<int64_t>(wave_m0) * dst_ld);
    const char* const res_u = GATE ? reinterpret_cast<const char*>(p.resid + static_cast<int64_t>(wave_m0) * p.ldresid + wave_n0) : nullptr;
    Vec16<bf16_t> rs[2][NACC], gs[2][GATE && EDGE ? NACC : 1];
    auto request_resid = [&](int i) {
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            if (EDGE) {   // past the end: values of the last valid row or the first column, not stored
                const int r = min(i * 16 + srow[a], rows_valid - 1), ch = (a * 64 + lane) % C_CH;
                rs[i & 1][a] = *reinterpret_cast<const Vec16<bf16_t>*>(res_u + static_cast<int64_t>(r) * p.ldresid * 2 + (wave_n0 + ch * 8 < p.N ? ch * 16 : 0));
                gs[i & 1][EDGE ? a : 0] = ld16(p.gate + static_cast<int64_t>((wave_m0 + r) / p.rows_per_batch) * p.gate_stride + wave_n0 + (wave_n0 + ch * 8 < p.N ? ch * 8 : 0));
            } else {
                rs[i & 1][a] = *reinterpret_cast<const Vec16<bf16_t>*>(res_u + static_cast<int64_t>(i) * 16 * p.ldresid * 2 + res_lane[a]);
            }
        }
    };
    if (GATE) request_resid(0);

#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        if (GATE) {
            if (i + 1 < ROWS) request_resid(i + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        char* const blk = cw + (i & 1) * (16 * C_PITCH);
#pragma unroll
        for (int q = 0; q < FN; ++q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = acc[i][q][e] + bv[q][e];
                if (GELU) v[e] = tanh_gelu_fast(v[e]);
            }
            *reinterpret_cast<u32x2*>(blk + waddr + q * 32) = pack4_bf16(v[0], v[1], v[2], v[3]);
        }
        __builtin_amdgcn_wave_barrier();   // LDS operations of one wave complete in order
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            const bool in = (SEGS % 64 == 0 || a * 64 + lane < SEGS) && (!EDGE || (i * 16 + srow[a] < rows_valid && wave_n0 + ((a * 64 + lane) % C_CH) * 8 < p.N));
            if (SEGS % 64 != 0 && a * 64 + lane >= SEGS) continue;
            Vec16<bf16_t> y = *reinterpret_cast<const Vec16<bf16_t>*>(blk + raddr[a]);
            if (GATE) {
                const Vec16<bf16_t> r = rs[i & 1][a];
                const Vec16<bf16_t> g = EDGE ? gs[i & 1][EDGE ? a : 0] : gt[EDGE ? 0 : a];
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const float y0 = bf2f(r.v[e]) + bf2f(f2bf(bf2f(g.v[e]) * bf2f(y.v[e])));
                    const float y1 = bf2f(r.v[e + 1]) + bf2f(f2bf(bf2f(g.v[e + 1]) * bf2f(y.v[e + 1])));
                    const uint32_t w = pack2_bf16(y0, y1);
                    y.v[e] = static_cast<bf16_t>(w & 0xffffu);
                    y.v[e + 1] = static_cast<bf16_t>(w >> 16);
                }
            }
            if (in) *reinterpret_cast<Vec16<bf16_t>*>(dst_u + static_cast<int64_t>(i) * 16 * dst_ld * 2 + dst_lane[a]) = y;
        }
    }
}

// Epilogue for what the branch-free forms cannot express: columns of any number and alignment, split_n and
// act_begin anywhere, GELU in front of a gate, rows any distance apart. The steps are those of
// gemm_epilogue_rect, decided per segment of 8 columns or per column. ROWS of the wave's FM fragment rows from `row0` on.
template <int FM, int FN, int ROWS>
__device__ __forceinline__ void gemm_epilogue_checked(const GemmParams& p, f32x4 (&acc)[ROWS][FN], char* lds, int m0, int n0, int row0, int wave, int lane) {
    constexpr int WCOLS = 16 * FN, C_CH = WCOLS / 8, C_PITCH = WCOLS * 2 + 16;
    constexpr int SEGS = 16 * C_CH;
    const int wm = wave >> 1, wn = wave & 1;
    const int frow = lane & 15, fq = lane >> 4;            // accumulator: row frow of a 16-row fragment, columns fq*4..+3
    char* cw = lds + wave * (2 * 16 * C_PITCH);
    const int wave_n0 = n0 + wn * WCOLS;
    const int wave_m0 = m0 + wm * (16 * FM) + row0 * 16;

    float bv[FN][4];
    if (p.bias != nullptr && p.bias_vec) {
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.bias), 0, p.N * 2, kRsrcFlags);
#pragma unroll
        for (int q = 0; q < FN; ++q) {
            const u32x2 raw = __builtin_amdgcn_raw_buffer_load_b64(rb, (wave_n0 + q * 16 + fq * 4) * 2, 0, 0);
            bv[q][0] = __uint_as_float(raw.x << 16);
            bv[q][1] = __uint_as_float(raw.x & 0xffff0000u);
            bv[q][2] = __uint_as_float(raw.y << 16);
            bv[q][3] = __uint_as_float(raw.y & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int q = 0; q < FN; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = wave_n0 + q * 16 + fq * 4 + e;
                bv[q][e] = (p.bias != nullptr && n < p.N) ? bf2f(p.bias[n]) : 0.0f;
            }
    }
    const bool gelu_all = p.act == FLUX_ACT_GELU_TANH && wave_n0 >= p.act_begin;
    const bool gelu_some = p.act == FLUX_ACT_GELU_TANH && !gelu_all && wave_n0 + WCOLS > p.act_begin;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        char* const blk = cw + (i & 1) * (16 * C_PITCH);
#pragma unroll
        for (int q = 0; q < FN; ++q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[i][q][e] + bv[q][e];
            if (gelu_all) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = tanh_gelu_fast(v[e]);
            } else if (gelu_some) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (wave_n0 + q * 16 + fq * 4 + e >= p.act_begin) v[e] = tanh_gelu_fast(v[e]);
            }
            *reinterpret_cast<u32x2*>(blk + frow * C_PITCH + fq * 8 + q * 32) = pack4_bf16(v[0], v[1], v[2], v[3]);
        }
        __builtin_amdgcn_wave_barrier();  // LDS operations of one wave complete in order
#pragma unroll
        for (int a = 0; a < (SEGS + 63) / 64; ++a) {
            const int seg = a * 64 + lane, row = seg / C_CH, ch = seg % C_CH;
            if (SEGS % 64 != 0 && seg >= SEGS) continue;
            const int m = wave_m0 + i * 16 + row, n = wave_n0 + ch * 8;
            Vec16<bf16_t> y = *reinterpret_cast<const Vec16<bf16_t>*>(blk + row * C_PITCH + ch * 16);
            if (m >= p.M || n >= p.N) continue;
            const bool full = p.vec_io && n + 8 <= p.N;
            if (p.gate != nullptr) {
                const bf16_t* gp = p.gate + static_cast<int64_t>(m / p.rows_per_batch) * p.gate_stride + n;
                const bf16_t* rp = p.resid + static_cast<int64_t>(m) * p.ldresid + n;
                if (full) {
                    Vec16<bf16_t> gt = ld16(gp), rs = ld16(rp);
#pragma unroll
                    for (int e = 0; e < 8; ++e) y.v[e] = f2bf(bf2f(rs.v[e]) + bf2f(f2bf(bf2f(gt.v[e]) * bf2f(y.v[e]))));
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (n + e < p.N) y.v[e] = f2bf(bf2f(rp[e]) + bf2f(f2bf(bf2f(gp[e]) * bf2f(y.v[e]))));
                }
            }
            if (full && (n + 8 <= p.split_n || n >= p.split_n)) {
                bf16_t* dst = n < p.split_n ? p.Y + static_cast<int64_t>(m) * p.ldy + n
                                            : p.Y2 + static_cast<int64_t>(m) * p.ldy2 + (n - p.split_n + p.y2_col0);
                st16(dst, y);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int ne = n + e;
                    if (ne < p.N) {
                        bf16_t* dst = ne < p.split_n ? p.Y + static_cast<int64_t>(m) * p.ldy + ne
                                                     : p.Y2 + static_cast<int64_t>(m) * p.ldy2 + (ne - p.split_n + p.y2_col0);
                        *dst = y.v[e];
                    }
                }
            }
        }
    }
}

// CHECKED: the tile has the checked epilogue too, for calls that carry p.checked.
template <int FM, int FN, int ROWS, bool CHECKED>
__device__ __forceinline__ void gemm_finish_rect(const GemmParams& p, f32x4 (&acc)[ROWS][FN], char* lds, int m0, int n0, int row0, int wave, int lane) {
    constexpr int BM = 32 * FM, WCOLS = 16 * FN;
    const int wave_n0 = n0 + (wave & 1) * WCOLS;
    if constexpr (CHECKED) {
        if (p.checked) return gemm_epilogue_checked<FM, FN, ROWS>(p, acc, lds, m0, n0, row0, wave, lane);
    }
    const bool gelu = p.act == FLUX_ACT_GELU_TANH && wave_n0 >= p.act_begin;
    const bool edge = m0 + BM > p.M || n0 + 32 * FN > p.N || (p.gate != nullptr && m0 / p.rows_per_batch != (m0 + BM - 1) / p.rows_per_batch);
    if constexpr (FN == 8 && ROWS > 1) {
        if (wave_n0 < p.qk_cols) {
            const bool ragged = m0 + BM > p.M || m0 / p.qk_seq_len != (m0 + BM - 1) / p.qk_seq_len;
            if (ragged) gemm_epilogue_qk<FM, FN / 2, ROWS, true>(p, acc, lds, m0, n0, row0, wave, lane);
            else gemm_epilogue_qk<FM, FN / 2, ROWS, false>(p, acc, lds, m0, n0, row0, wave, lane);
            return;
        }
    }
    if (p.gate != nullptr) {   // (the host admits a gate without GELU only)
        if (edge) gemm_epilogue_rect<FM, FN, ROWS, false, true, true>(p, acc, lds, m0, n0, row0, wave, lane);
        else gemm_epilogue_rect<FM, FN, ROWS, false, true, false>(p, acc, lds, m0, n0, row0, wave, lane);
    } else if (gelu) {
        if (edge) gemm_epilogue_rect<FM, FN, ROWS, true, false, true>(p, acc, lds, m0, n0, row0, wave, lane);
        else gemm_epilogue_rect<FM, FN, ROWS, true, false, false>(p, acc, lds, m0, n0, row0, wave, lane);
    } else {
        if (edge) gemm_epilogue_rect<FM, FN, ROWS, false, false, true>(p, acc, lds, m0, n0, row0, wave, lane);
        else gemm_epilogue_rect<FM, FN, ROWS, false, false, false>(p, acc, lds, m0, n0, row0, wave, lane);
    }
}

// Whether a program is unlikely to find a launch's weights in the Infinity Cache: they are more than a third of it.
inline bool weights_from_hbm(const GemmSet& g) { return static_cast<int64_t>(g.n) * g.p[0].N * g.p[0].K * 2 > (int64_t{256} << 20) / 3; }

inline GemmLaunch make_launch(const GemmSet& g, int bm, int bn) {
    GemmLaunch L;
    const GemmParams& p = g.p[0];
    L.p[0] = p;
    L.p[1] = g.p[g.n - 1];
    L.tiles_m0 = L.tiles_m = (p.M + bm - 1) / bm;
    if (g.n > 1) L.tiles_m += (g.p[1].M + bm - 1) / bm;
    L.tiles_n = (p.N + bn - 1) / bn;
    L.group_m = 4;
    L.splits = 1;
    L.slabs_per_split = (p.K + 63) / 64;
    L.take_turns = false;
    L.partial = nullptr;
    return L;
}
inline unsigned grid_of(const GemmLaunch& L) { return static_cast<unsigned>((L.tiles_m * L.tiles_n * L.splits + 7) / 8 * 8); }

// Eight-wave tiles (gemm_pair.hip). K range in `splits` parts, which then need `partial`.
void launch_pair_tiles(int fm, int fn, const GemmSet& g, int splits, float* partial, hipStream_t st);

}  // namespace flux
