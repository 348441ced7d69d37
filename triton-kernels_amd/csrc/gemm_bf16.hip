// Linear layer on the matrix cores:  Y = epilogue(A[M,K] * W[N,K]^T), bf16 operands, fp32 accumulate.
//
// Both operands are K-contiguous, which is exactly what v_mfma_f32_16x16x32_bf16 wants: every lane
// feeds 8 consecutive k of one row. A workgroup of four waves (2 x 2) owns a (64*MI) x (64*MI) tile
// of Y and each wave a (32*MI) x (32*MI) sub-tile kept as (2*MI)^2 accumulators of 16x16. (The
// 16x16x32 shape moves half the accumulator registers per flop of 32x32x16; on a chip that runs
// this kernel at its power limit that is worth more than the extra instruction issues.) The K loop
// moves 64-wide slabs of A and W through a five-unit LDS ring (see the kernel) straight from buffer
// loads that write LDS (no register staging).
//
// LDS slab layout: row r of the slab is 128 bytes = eight 16-byte chunks; chunk c is stored at
// position c ^ ((r >> 1) & 7). LDS on gfx950 has 64 banks of 4 bytes, so a ds_read_b128 is served 16
// lanes (256 bytes) per clock: the 16 lanes that read the same logical chunk of 16 consecutive rows
// land on 2 (row parity) x 8 (position) = 16 different 16-byte bank groups, conflict-free. The
// writer side fills whole rows, also conflict-free.
//
// The MFMA takes W as its "A" operand and the activations as its "B" operand, so the accumulator
// of a lane holds one activation row m and runs of 4 consecutive output columns n: bias and GELU
// are applied there in fp32 and the result is rounded once; the bf16 tile goes through LDS once
// more and leaves as full 16-byte row segments, where the optional gated residual is applied.
#include "gemm_common.h"
#include "gemm_rows.h"
#include <limits.h>
#include <stdlib.h>
#include <algorithm>

namespace flux {

// Branch-free epilogue for interior tiles whose outputs (and residual operands) are 16-byte
// addressable and whose columns all go to one destination. GELU is all-or-nothing for the wave.
// Everything lane-dependent is computed once; per store only a wave-uniform row offset changes, so
// the stores use a scalar base plus a 32-bit lane offset.
template <int MI, int NJ, bool GELU, bool GATE>
__device__ __forceinline__ void gemm_epilogue_fast(const GemmParams& p, f32x4 (&acc)[2 * MI][2 * NJ], char* lds, int m0, int n0,
                                                   int wave, int lane) {
    constexpr int WROWS = 32 * MI, WCOLS = 32 * NJ;
    constexpr int C_PITCH = WCOLS * 2, C_CH = WCOLS / 8;
    constexpr int RPI = 64 / C_CH;      // rows per wave-wide 16-byte access
    constexpr int NIT = 32 / RPI;       // accesses per 32-row block
    constexpr int NQ = 2 * NJ;          // column quads of a lane: one per 16-column fragment
    const int wm = wave >> 1, wn = wave & 1;
    const int frow = lane & 15, fq = lane >> 4;
    char* cw = lds + wave * (WROWS * C_PITCH);
    const int wave_n0 = n0 + wn * WCOLS;
    const int wave_m0 = m0 + wm * WROWS;

    float bv[NQ][4];
    if (p.bias != nullptr) {
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.bias), 0, p.N * 2, kRsrcFlags);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const u32x2 raw = __builtin_amdgcn_raw_buffer_load_b64(rb, (wave_n0 + q * 16 + fq * 4) * 2, 0, 0);
            bv[q][0] = __uint_as_float(raw.x << 16);
            bv[q][1] = __uint_as_float(raw.x & 0xffff0000u);
            bv[q][2] = __uint_as_float(raw.y << 16);
            bv[q][3] = __uint_as_float(raw.y & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[q][e] = 0.0f;
    }

    int waddr[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) waddr[q] = frow * C_PITCH + (((q * 2 + (fq >> 1)) ^ (frow & (C_CH - 1))) * 16) + (fq & 1) * 8;
    const int rrow = lane / C_CH, rch = lane % C_CH;
    // read address for access `it` of a block: row = it*RPI + rrow; the swizzle term repeats every 16 rows
    constexpr int NSW = (16 / RPI) < NIT ? (16 / RPI) : NIT;
    int raddr[NSW];
#pragma unroll
    for (int t = 0; t < NSW; ++t) {
        const int row = t * RPI + rrow;
        raddr[t] = row * C_PITCH + ((rch ^ (row & (C_CH - 1))) * 16);
    }

    const bool to_y = wave_n0 < p.split_n;
    char* dst_u = reinterpret_cast<char*>(to_y ? p.Y + wave_n0 : p.Y2 + (wave_n0 - p.split_n + p.y2_col0));
    const int64_t dst_ld = (to_y ? p.ldy : p.ldy2) * 2;            // bytes
    const uint32_t dst_lane = static_cast<uint32_t>(rrow * dst_ld + rch * 16);
    // Gated residual: the rows of resid this lane adds to are requested a whole 32-row block ahead,
    // into the other half of rs, so that they land while the block in front is converted and stored.
    // (Requested where they are used, every 16-byte store waited for a load round trip of its own,
    // and, the memory counter being in-order, for the store in front of it: 32 round trips in a row
    // per wave.) The tile lies inside one batch element (the caller checks), so the gate vector of
    // this lane's eight columns is loaded once.
    const char* res_u = nullptr;
    uint32_t res_lane = 0;
    Vec16<bf16_t> gt;
    Vec16<bf16_t> rs[2][NIT];
    auto request_resid = [&](int i) {
#pragma unroll
        for (int it = 0; it < NIT; ++it)
            rs[i & 1][it] = *reinterpret_cast<const Vec16<bf16_t>*>(res_u + static_cast<int64_t>(wave_m0 + i * 32 + it * RPI) * p.ldresid * 2 + res_lane);
    };
    if (GATE) {
        res_u = reinterpret_cast<const char*>(p.resid + wave_n0);
        res_lane = static_cast<uint32_t>(rrow * p.ldresid * 2 + rch * 16);
        gt = ld16(p.gate + static_cast<int64_t>(m0 / p.rows_per_batch) * p.gate_stride + wave_n0 + rch * 8);
        request_resid(0);
    }

#pragma unroll
    for (int i = 0; i < MI; ++i) {
        if (GATE) {
            if (i + 1 < MI) request_resid(i + 1);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay in front of the conversion below
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = acc[2 * i + t][q][e] + bv[q][e];
                    if (GELU) v[e] = tanh_gelu_fast(v[e]);
                }
                *reinterpret_cast<u32x2*>(cw + (i * 32 + t * 16) * C_PITCH + waddr[q]) = pack4_bf16(v[0], v[1], v[2], v[3]);
            }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const int row_u = i * 32 + it * RPI;                 // wave-uniform part of the row
            Vec16<bf16_t> y = *reinterpret_cast<const Vec16<bf16_t>*>(cw + (i * 32 + (it / NSW) * NSW * RPI) * C_PITCH + raddr[it % NSW]);
            const int64_t m_u = wave_m0 + row_u;
            if (GATE) {
                const Vec16<bf16_t> r = rs[i & 1][it];
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const float y0 = bf2f(r.v[e]) + bf2f(f2bf(bf2f(gt.v[e]) * bf2f(y.v[e])));
                    const float y1 = bf2f(r.v[e + 1]) + bf2f(f2bf(bf2f(gt.v[e + 1]) * bf2f(y.v[e + 1])));
                    const uint32_t w = pack2_bf16(y0, y1);
                    y.v[e] = static_cast<bf16_t>(w & 0xffffu);
                    y.v[e + 1] = static_cast<bf16_t>(w >> 16);
                }
            }
            *reinterpret_cast<Vec16<bf16_t>*>(dst_u + m_u * dst_ld + dst_lane) = y;
        }
    }
}

template <int MI, int NJ>
__device__ __forceinline__ void gemm_epilogue(const GemmParams& p, f32x4 (&acc)[2 * MI][2 * NJ], char* lds, int m0, int n0,
                                              int wave, int lane) {
    constexpr int BM = 64 * MI, BN = 64 * NJ, WCOLS = 32 * NJ;
    const int wave_n0 = n0 + (wave & 1) * WCOLS;
    const bool gelu_all = p.act == FLUX_ACT_GELU_TANH && wave_n0 >= p.act_begin;
    const bool gelu_none = p.act != FLUX_ACT_GELU_TANH || wave_n0 + WCOLS <= p.act_begin;
    if constexpr (NJ == 4) {
        if (wave_n0 < p.qk_cols) {   // the host admits the fusion only when the q/k columns are whole tiles
            const bool ragged = m0 + BM > p.M || m0 / p.qk_seq_len != (m0 + BM - 1) / p.qk_seq_len;
            if (ragged) gemm_epilogue_qk<2 * MI, NJ, 2 * MI, true>(p, acc, lds, m0, n0, 0, wave, lane);
            else gemm_epilogue_qk<2 * MI, NJ, 2 * MI, false>(p, acc, lds, m0, n0, 0, wave, lane);
            return;
        }
    }
    // (with a gate: the fast path loads one gate vector per tile, so the tile must not span batch elements)
    const bool fast = p.vec_io && m0 + BM <= p.M && n0 + BN <= p.N && (gelu_all || gelu_none) &&
                      (p.gate == nullptr || m0 / p.rows_per_batch == (m0 + BM - 1) / p.rows_per_batch) &&
                      (wave_n0 + WCOLS <= p.split_n || wave_n0 >= p.split_n) && (p.bias == nullptr || p.bias_vec) &&
                      static_cast<int64_t>(BM) * p.ldy * 2 < 0x7fffffffLL && static_cast<int64_t>(BM) * p.ldy2 * 2 < 0x7fffffffLL &&
                      static_cast<int64_t>(BM) * p.ldresid * 2 < 0x7fffffffLL;
    if (fast) {
        if (p.gate != nullptr) {
            if (gelu_all) gemm_epilogue_fast<MI, NJ, true, true>(p, acc, lds, m0, n0, wave, lane);
            else gemm_epilogue_fast<MI, NJ, false, true>(p, acc, lds, m0, n0, wave, lane);
        } else {
            if (gelu_all) gemm_epilogue_fast<MI, NJ, true, false>(p, acc, lds, m0, n0, wave, lane);
            else gemm_epilogue_fast<MI, NJ, false, false>(p, acc, lds, m0, n0, wave, lane);
        }
    } else {
        gemm_epilogue_checked<2 * MI, 2 * NJ, 2 * MI>(p, acc, lds, m0, n0, 0, wave, lane);
    }
}

// ------------------------------------------------------------------------------------------------
// Tiled kernel: 64*MI x 64*MI output tile per workgroup of four waves (2 x 2, a wave owns
// 32*MI x 32*MI as (2*MI)^2 accumulators of v_mfma_f32_16x16x32_bf16), K in slabs of 64 = two MFMA
// steps of K = 32. With two whole-slab LDS stages the memory pipeline would drain at every barrier
// (the wait in front of it is for ALL outstanding loads). Here LDS is a ring of five units, a unit
// holding one operand's share of a slab (BM rows x 128 bytes): A(kt) lives in unit 2kt % 5 and
// W(kt) in unit (2kt+1) % 5. While slab kt is computed, slab kt+1 and A(kt+2) occupy the other
// three units. The barrier of slab kt sits a quarter into its last step; right behind it the unit
// of A(kt) is free and takes the loads of W(kt+2), one per slot, and the loads of A(kt+3) follow at
// an even pace in front of the next barrier. The wait in front of a barrier only covers W of the
// next slab: the loads of A two slabs ahead stay in flight across it. Every load has more than
// three quarters of a slab of MFMA time to land and the memory pipeline never runs empty.
//
//   slab kt :  step 0            step 1 = [MFMA x PER*BS] wait+barrier [rest, reads step 0 of kt+1]
//   loads   :  ...... A(kt+2) ......................      |  W(kt+2) x PU, one per slot
//
// Ring offsets are wave-uniform scalars that advance by two units per slab.
// ------------------------------------------------------------------------------------------------
// Multiplies the first ke K slabs of the tile at (m0, n0) into acc (cleared first). On return every
// buffer load of the wave has landed and all waves have passed a barrier, so the ring may be
// reused (the epilogue parks its bf16 blocks there).
template <int MI, bool KTAIL>
__device__ __forceinline__ void gemm_tile_slabs(const GemmParams& p, char* lds, int m0, int n0, int ke,
                                                f32x4 (&acc)[2 * MI][2 * MI]) {
    constexpr int NJ = MI;
    constexpr int FM = 2 * MI, FN = 2 * NJ;      // 16-row fragments per wave and side
    constexpr int BM = 64 * MI, BN = BM, BK = 64;
    constexpr int ROWB = BK * 2, KSUB = BK / 32;
    constexpr int UNIT = BM * ROWB, NU = 5;
    constexpr int PU = BM / 32;                  // buffer loads per thread per unit
    constexpr int NL = 2 * PU;                   // loads per group G(kt) = W(kt+1), A(kt+2)
    constexpr int WROWS = 32 * MI, WCOLS = 32 * NJ;
    constexpr int READS = FM + FN, MFMAS = FM * FN, PER = MFMAS / READS;
    constexpr int BS = READS / 4;                // slots of the last step in front of the barrier
    constexpr int NSLOT = KSUB * READS;          // issue slots per slab
    constexpr int GB = (KSUB - 1) * READS + BS;  // first slot behind the barrier
    constexpr int EARLY = PU;                    // W loads of a group, all issued right behind the previous slab's barrier
    static_assert(MFMAS % READS == 0 && KSUB == 2 && NSLOT == 2 * NL && NSLOT - GB >= PU, "schedule shape");
    static_assert(2 * (NSLOT - GB) >= READS, "the next slab's first fragments are read two per slot behind the barrier");
    static_assert(4 * WROWS * WCOLS * 2 <= NU * UNIT, "epilogue tile must fit the ring");
    (void)BN; (void)WCOLS;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // loader mapping: LDS slot (row = pass*32 + tid/8, position tid%8) holds logical chunk
    // position ^ ((row>>1)&7) of that row
    const int lrow = tid >> 3;
    const int lchunk = (tid & 7) ^ ((lrow >> 1) & 7);
    const int rows_a = min(p.M - m0, BM), rows_b = min(p.N - n0, BN);
    const int64_t a0 = row_of_a(p, m0);
    bf16_t* const base_a = const_cast<bf16_t*>(p.A + a0);
    bf16_t* const base_b = const_cast<bf16_t*>(p.W + static_cast<int64_t>(n0) * p.ldw);
    const int bytes_a = static_cast<int>((row_of_a(p, m0 + rows_a - 1) - a0 + p.K) * 2);
    const int bytes_b = static_cast<int>(((rows_b - 1) * p.ldw + p.K) * 2);
    uint32_t voff_a[PU], voff_b[PU];
#pragma unroll
    for (int i = 0; i < PU; ++i) {
        const int r = i * 32 + lrow;
        voff_a[i] = r < rows_a ? static_cast<uint32_t>((row_of_a(p, m0 + r) - a0 + lchunk * 8) * 2) : kOutOfRange;
        voff_b[i] = r < rows_b ? static_cast<uint32_t>((r * p.ldw + lchunk * 8) * 2) : kOutOfRange;
    }
    // the slab range ends at ke: everything from there on reads as zeros, like the K tail
    const int k_end = min(p.K, ke * BK);
    // Slabs past the end and the part of the last slab past K read as zeros. With a K tail (KTAIL)
    // that is "this thread's chunk starts at or past K" (K is a multiple of 8, so a chunk is all in
    // or all out) and the mask is a per-lane offset bit. Without one a slab is all in or all out,
    // the mask is wave-uniform and selects a buffer resource of zero records instead, which keeps
    // the vector ALU out of the loop.
    auto slab_mask = [&](int kt) -> uint32_t {
        if constexpr (KTAIL) return kt * BK + lchunk * 8 >= k_end ? kOutOfRange : 0u;
        else return kt * BK >= k_end ? kOutOfRange : 0u;
    };
    // ring offsets are wave-uniform byte offsets of a unit inside the ring
    auto load_a = [&](int uoff, int pass, int kt, uint32_t mask) {
        if constexpr (KTAIL) {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_a, 0, bytes_a, kRsrcFlags), lds + uoff + pass * 4096 + wave * 1024,
                       voff_a[pass] | mask, kt * ROWB);
        } else {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_a, 0, mask ? 0 : bytes_a, kRsrcFlags),
                       lds + uoff + pass * 4096 + wave * 1024, voff_a[pass], kt * ROWB);
        }
    };
    auto load_w = [&](int uoff, int pass, int kt, uint32_t mask) {
        if constexpr (KTAIL) {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_b, 0, bytes_b, kRsrcFlags), lds + uoff + pass * 4096 + wave * 1024,
                       voff_b[pass] | mask, kt * ROWB);
        } else {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_b, 0, mask ? 0 : bytes_b, kRsrcFlags),
                       lds + uoff + pass * 4096 + wave * 1024, voff_b[pass], kt * ROWB);
        }
    };

    // fragment addressing
    // v_mfma_f32_16x16x32_bf16 operand: lane holds row lane % 16, k = (lane / 16) * 8 .. +8 of a K=32 step
    const int frow = lane & 15, fq = lane >> 4;
    int koff_a[KSUB], koff_w[KSUB];
#pragma unroll
    for (int kk = 0; kk < KSUB; ++kk) {
        const int ko = ((kk * 4 + fq) ^ ((frow >> 1) & 7)) * 16;
        koff_a[kk] = (wm * WROWS + frow) * ROWB + ko;
        koff_w[kk] = (wn * WCOLS + frow) * ROWB + ko;
    }

#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

    bf16x8 xa[2][FM], wb[2][FN];
    // r-th fragment of K-step kk of the slab whose units start at ua / uw, in the order the MFMAs
    // first need them: x0, w0..w(FN-1), x1..x(FM-1)
    auto read_frag = [&](int buf, int ua, int uw, int kk, int r) {
        const char* pa = lds + (ua + koff_a[kk]);
        const char* pw = lds + (uw + koff_w[kk]);
        if (r == 0) xa[buf][0] = *reinterpret_cast<const bf16x8*>(pa);
        else if (r <= FN) wb[buf][r - 1] = *reinterpret_cast<const bf16x8*>(pw + (r - 1) * 16 * ROWB);
        else xa[buf][r - FN] = *reinterpret_cast<const bf16x8*>(pa + (r - FN) * 16 * ROWB);
    };
    auto mfma_one = [&](int buf, int idx) {
        // boustrophedon over the accumulator grid: from one MFMA to the next only one of the two
        // operands changes, also at the end of a row (about 1 % less time at the power limit)
        const int i = idx / FN, j = (i & 1) ? FN - 1 - idx % FN : idx % FN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[buf][j], xa[buf][i], acc[i][j], 0, 0, 0);
    };

    // ua/uw: units of slab kt, ua1/uw1: of slab kt+1, ua2: of A(kt+2); W(kt+2) takes over ua once
    // the barrier has retired it. m2: load mask of slab kt+2; the mask of slab kt+3 is
    // worked out in the shadow of an MFMA so that the loop back-edge carries register moves only.
    auto slab = [&](int kt, int ua, int uw, int ua1, int uw1, int ua2, uint32_t m2, uint32_t& m3) {
        const int uw2 = ua;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < NSLOT; ++s) {
            const int stp = s / READS, r = s % READS;
            if (s == GB) {
                wait_loads_and_barrier<PU>();  // slab kt+1 is complete in LDS; this slab's units are free
                __builtin_amdgcn_sched_barrier(0);
            }
            auto slot_reads = [&]() {
                if (stp < KSUB - 1) {
                    read_frag((stp & 1) ^ 1, ua, uw, stp + 1, r);
                } else if (r >= BS) {
                    // two per slot: the last one is requested a few MFMAs before the slab ends, so the
                    // wait at the top of the next slab finds it done
                    const int lo = 2 * (r - BS);
                    for (int f = lo; f < lo + 2 && f < READS; ++f) read_frag(0, ua1, uw1, 0, f);
                }
            };
            // one memory instruction per MFMA interval: the fragment read goes in front of the slot's
            // first MFMA, the buffer load behind it. The slab's first MFMA waits for the fragments
            // requested at the end of the previous slab, and that wait is for every outstanding LDS
            // read: the first read of this slab is therefore issued behind it, not in front.
            if (s != 0) slot_reads();
            mfma_one(stp & 1, r * PER);
            if (s == 0) {
                __builtin_amdgcn_sched_barrier(0);
                slot_reads();
            }
            if (s == 1) m3 = slab_mask(kt + 3);
            __builtin_amdgcn_sched_barrier(0);
            if (s < GB) {
                // A(kt+2): PU loads spread evenly over the slots in front of the barrier
#pragma unroll
                for (int i = 0; i < PU; ++i)
                    if ((i * GB) / PU == s) load_a(ua2, i, kt + 2, m2);
            } else if (s - GB < PU) {
                load_w(uw2, s - GB, kt + 2, m2);   // W(kt+2): one per slot right behind the barrier
            }
#pragma unroll
            for (int m = 1; m < PER; ++m) mfma_one(stp & 1, r * PER + m);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // Prologue: slab 0, A(1) and the first loads of G(0); slab 0 must have landed, the rest flies on.
    {
        const uint32_t k0 = slab_mask(0), k1 = slab_mask(1);
#pragma unroll
        for (int i = 0; i < PU; ++i) load_a(0, i, 0, k0);
#pragma unroll
        for (int i = 0; i < PU; ++i) load_w(UNIT, i, 0, k0);
#pragma unroll
        for (int i = 0; i < PU; ++i) load_a(2 * UNIT, i, 1, k1);
#pragma unroll
        for (int i = 0; i < EARLY; ++i) load_w(3 * UNIT, i, 1, k1);
        wait_loads_and_barrier<PU + EARLY>();
#pragma unroll
        for (int r = 0; r < READS; ++r) read_frag(0, 0, UNIT, 0, r);
        __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(EARLY <= PU, "loads behind the barrier must all belong to W");

    {
        int ua = 0, uw = UNIT, ua1 = 2 * UNIT, uw1 = 3 * UNIT, ua2 = 4 * UNIT;
        uint32_t m2 = slab_mask(2);
        for (int kt = 0; kt < ke; ++kt) {
            uint32_t m3;
            slab(kt, ua, uw, ua1, uw1, ua2, m2, m3);
            // the ring advances by two units
            const int t0 = ua, t1 = uw;
            ua = ua1; uw = uw1; ua1 = ua2; uw1 = t0; ua2 = t1;
            m2 = m3;
        }
    }
    // The last slab's trailing loads were masked (they move no data but still write zeros to LDS):
    // retire them before the epilogue reuses the ring.
    wait_vmem_all();
    __syncthreads();
}


// TWO: the launch may hold two products, whose parameters are taken by reference (a copy, see product_of_tile, does
// not fit the scalar registers of the 256-wide tile); the form for one reads them as plain kernel arguments.
template <int MI, bool KTAIL, bool TWO>
__global__ __launch_bounds__(kGemmThreads) void gemm_nt_ring_kernel(GemmLaunch L) {
    constexpr int BM = 64 * MI, BK = 64, NU = 5, UNIT = BM * BK * 2;
    __shared__ __attribute__((aligned(1024))) char lds[NU * UNIT];
    int tm, tn;
    if (L.p[0].qk_cols > 0 ? !tile_of_block_qk(L, BM, tm, tn) : !tile_of_block(L, tm, tn)) return;
    const GemmParams& p = L.p[TWO ? product_of_tile(L, tm) : 0];
    const int m0 = tm * BM, n0 = tn * BM;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 acc[2 * MI][2 * MI];
    gemm_tile_slabs<MI, KTAIL>(p, lds, m0, n0, (p.K + BK - 1) / BK, acc);
    gemm_epilogue<MI, MI>(p, acc, lds, m0, n0, wave, lane);
}

// ------------------------------------------------------------------------------------------------
// Rectangular tiles: (32*FM) x (32*FN) per workgroup, a wave owns (16*FM) x (16*FN) as FM x FN
// accumulators. One workgroup per CU means a launch costs whole rounds of 256 tiles; 4608 x 3072
// (linear2 of the Flux block) is 216 tiles of 256 x 256, 0.84 of a round with 40 CUs idle, but
// exactly 256 tiles of 288 x 192 (FM = 9, FN = 6: 216 accumulation registers). The main loop is the
// one above with the two operands' slabs in rings of their own, because their units now differ in
// size: three units of A (BM rows x 128 bytes) and two of W (BN rows), 156 KB. While slab kt is
// multiplied, A(kt+1), W(kt+1) and A(kt+2) occupy the other units; behind the barrier of slab kt the
// unit of W(kt) takes W(kt+2), and the loads of A(kt+3) go into the unit of A(kt) in front of the
// next barrier. A step has FM + FN fragment reads for FM * FN MFMAs, which no longer divide: slot r
// issues MFMAs [r * MFMAS / READS, (r + 1) * MFMAS / READS).
// Rows past M or N read as zeros and are not stored.
// ------------------------------------------------------------------------------------------------
template <int FM, int FN, bool KTAIL>
__device__ __forceinline__ void gemm_rect_slabs(const GemmParams& p, char* lds, int m0, int n0, int ke, f32x4 (&acc)[FM][FN]) {
    constexpr int BM = 32 * FM, BN = 32 * FN, BK = 64;
    constexpr int ROWB = BK * 2, KSUB = BK / 32;
    constexpr int UNIT_A = BM * ROWB, UNIT_W = BN * ROWB, W0 = 3 * UNIT_A;   // W ring behind the A ring
    constexpr int PA = BM / 32, PW = BN / 32;    // buffer loads per thread per unit of A / W
    constexpr int WROWS = 16 * FM, WCOLS = 16 * FN;
    constexpr int READS = FM + FN, MFMAS = FM * FN;
    constexpr int BS = READS / 4;                // slots of the last step in front of the barrier
    constexpr int NSLOT = KSUB * READS;          // issue slots per slab
    constexpr int GB = (KSUB - 1) * READS + BS;  // first slot behind the barrier
    static_assert(KSUB == 2 && GB >= PA && NSLOT - GB >= PW && MFMAS >= READS, "schedule shape");
    static_assert(2 * (NSLOT - GB) >= READS, "the next slab's first fragments are read two per slot behind the barrier");
    static_assert(BM % 32 == 0 && BN % 32 == 0 && (WROWS / 2) % 8 == 0 && (WCOLS / 2) % 8 == 0, "row swizzle must not see the wave offset");
    static_assert(3 * UNIT_A + 2 * UNIT_W <= 160 * 1024, "rings must fit the LDS");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // loader mapping as in the square kernel: LDS slot (row = pass*32 + tid/8, position tid%8) holds
    // logical chunk position ^ ((row>>1)&7) of that row
    const int lrow = tid >> 3;
    const int lchunk = (tid & 7) ^ ((lrow >> 1) & 7);
    const int rows_a = min(p.M - m0, BM), rows_b = min(p.N - n0, BN);
    const int64_t a0 = row_of_a(p, m0);
    bf16_t* const base_a = const_cast<bf16_t*>(p.A + a0);
    bf16_t* const base_b = const_cast<bf16_t*>(p.W + static_cast<int64_t>(n0) * p.ldw);
    const int bytes_a = static_cast<int>((row_of_a(p, m0 + rows_a - 1) - a0 + p.K) * 2);
    const int bytes_b = static_cast<int>(((rows_b - 1) * p.ldw + p.K) * 2);
    uint32_t voff_a[PA], voff_b[PW];
#pragma unroll
    for (int i = 0; i < PA; ++i) voff_a[i] = i * 32 + lrow < rows_a ? static_cast<uint32_t>((row_of_a(p, m0 + i * 32 + lrow) - a0 + lchunk * 8) * 2) : kOutOfRange;
#pragma unroll
    for (int i = 0; i < PW; ++i) voff_b[i] = i * 32 + lrow >= rows_b ? kOutOfRange : static_cast<uint32_t>(((i * 32 + lrow) * p.ldw + lchunk * 8) * 2);
    const int k_end = min(p.K, ke * BK);
    auto slab_mask = [&](int kt) -> uint32_t {
        if constexpr (KTAIL) return kt * BK + lchunk * 8 >= k_end ? kOutOfRange : 0u;
        else return kt * BK >= k_end ? kOutOfRange : 0u;
    };
    auto load_a = [&](int uoff, int pass, int kt, uint32_t mask) {
        if constexpr (KTAIL) {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_a, 0, bytes_a, kRsrcFlags), lds + uoff + pass * 4096 + wave * 1024,
                       voff_a[pass] | mask, kt * ROWB);
        } else {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_a, 0, mask ? 0 : bytes_a, kRsrcFlags),
                       lds + uoff + pass * 4096 + wave * 1024, voff_a[pass], kt * ROWB);
        }
    };
    auto load_w = [&](int uoff, int pass, int kt, uint32_t mask) {
        if constexpr (KTAIL) {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_b, 0, bytes_b, kRsrcFlags), lds + W0 + uoff + pass * 4096 + wave * 1024,
                       voff_b[pass] | mask, kt * ROWB);
        } else {
            load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_b, 0, mask ? 0 : bytes_b, kRsrcFlags),
                       lds + W0 + uoff + pass * 4096 + wave * 1024, voff_b[pass], kt * ROWB);
        }
    };

    const int frow = lane & 15, fq = lane >> 4;
    int koff_a[KSUB], koff_w[KSUB];
#pragma unroll
    for (int kk = 0; kk < KSUB; ++kk) {
        const int ko = ((kk * 4 + fq) ^ ((frow >> 1) & 7)) * 16;
        koff_a[kk] = (wm * WROWS + frow) * ROWB + ko;
        koff_w[kk] = W0 + (wn * WCOLS + frow) * ROWB + ko;
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

    bf16x8 xa[2][FM], wb[2][FN];
    auto read_frag = [&](int buf, int ua, int uw, int kk, int r) {
        const char* pa = lds + (ua + koff_a[kk]);
        const char* pw = lds + (uw + koff_w[kk]);
        if (r == 0) xa[buf][0] = *reinterpret_cast<const bf16x8*>(pa);
        else if (r <= FN) wb[buf][r - 1] = *reinterpret_cast<const bf16x8*>(pw + (r - 1) * 16 * ROWB);
        else xa[buf][r - FN] = *reinterpret_cast<const bf16x8*>(pa + (r - FN) * 16 * ROWB);
    };
    auto mfma_one = [&](int buf, int idx) {
        const int i = idx / FN, j = (i & 1) ? FN - 1 - idx % FN : idx % FN;   // boustrophedon, as above
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[buf][j], xa[buf][i], acc[i][j], 0, 0, 0);
    };

    // ua, ua1, ua2: units of A(kt), A(kt+1), A(kt+2); uw, uw1: of W(kt), W(kt+1); W(kt+2) takes over uw
    // behind the barrier
    auto slab = [&](int kt, int ua, int ua1, int ua2, int uw, int uw1, uint32_t m2, uint32_t& m3) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < NSLOT; ++s) {
            const int stp = s / READS, r = s % READS;
            const int lo = r * MFMAS / READS, hi = (r + 1) * MFMAS / READS;
            if (s == GB) {
                wait_loads_and_barrier<PA>();  // W(kt+1) has landed (A(kt+1) before it); this slab's units are free
                __builtin_amdgcn_sched_barrier(0);
            }
            auto slot_reads = [&]() {
                if (stp < KSUB - 1) {
                    read_frag((stp & 1) ^ 1, ua, uw, stp + 1, r);
                } else if (r >= BS) {
                    const int f0 = 2 * (r - BS);
                    for (int f = f0; f < f0 + 2 && f < READS; ++f) read_frag(0, ua1, uw1, 0, f);
                }
            };
            if (s != 0) slot_reads();
            mfma_one(stp & 1, lo);
            if (s == 0) {
                __builtin_amdgcn_sched_barrier(0);
                slot_reads();
            }
            if (s == 1) m3 = slab_mask(kt + 3);
            __builtin_amdgcn_sched_barrier(0);
            if (s < GB) {
#pragma unroll
                for (int i = 0; i < PA; ++i)
                    if ((i * GB) / PA == s) load_a(ua2, i, kt + 2, m2);
            } else if (s - GB < PW) {
                load_w(uw, s - GB, kt + 2, m2);
            }
#pragma unroll
            for (int m = lo + 1; m < hi; ++m) mfma_one(stp & 1, m);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    {
        const uint32_t k0 = slab_mask(0), k1 = slab_mask(1);
#pragma unroll
        for (int i = 0; i < PA; ++i) load_a(0, i, 0, k0);
#pragma unroll
        for (int i = 0; i < PW; ++i) load_w(0, i, 0, k0);
#pragma unroll
        for (int i = 0; i < PA; ++i) load_a(UNIT_A, i, 1, k1);
#pragma unroll
        for (int i = 0; i < PW; ++i) load_w(UNIT_W, i, 1, k1);
        wait_loads_and_barrier<PA + PW>();
#pragma unroll
        for (int r = 0; r < READS; ++r) read_frag(0, 0, 0, 0, r);
        __builtin_amdgcn_sched_barrier(0);
    }
    {
        int ua = 0, ua1 = UNIT_A, ua2 = 2 * UNIT_A, uw = 0, uw1 = UNIT_W;
        uint32_t m2 = slab_mask(2);
        for (int kt = 0; kt < ke; ++kt) {
            uint32_t m3;
            slab(kt, ua, ua1, ua2, uw, uw1, m2, m3);
            const int t0 = ua, t1 = uw;
            ua = ua1; ua1 = ua2; ua2 = t0;
            uw = uw1; uw1 = t1;
            m2 = m3;
        }
    }
    wait_vmem_all();
    __syncthreads();
}

template <int FM, int FN, bool KTAIL>
__global__ __launch_bounds__(kGemmThreads) void gemm_nt_rect_kernel(GemmLaunch L) {
    constexpr int BM = 32 * FM, BN = 32 * FN, BK = 64;
    __shared__ __attribute__((aligned(1024))) char lds[(3 * BM + 2 * BN) * BK * 2];
    int tm, tn;
    if (FN == 8 && L.p[0].qk_cols > 0 ? !tile_of_block_qk(L, BN, tm, tn) : !tile_of_block(L, tm, tn)) return;
    const GemmParams p = L.p[product_of_tile(L, tm)];
    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 acc[FM][FN];
    gemm_rect_slabs<FM, FN, KTAIL>(p, lds, m0, n0, (p.K + BK - 1) / BK, acc);
    gemm_finish_rect<FM, FN, FM, false>(p, acc, lds, m0, n0, 0, wave, lane);
}

template <int MM, bool SILU_LDS, int U, bool EXACT, bool ONCE>
__global__ __launch_bounds__(256) void gemv_small_m_kernel(GemmSet g) {
    extern __shared__ __attribute__((aligned(16))) char act_lds[];
    const GemmParams p = g.p[blockIdx.y];
    gemv_small_m<MM, SILU_LDS, U, EXACT, ONCE>(p, static_cast<int>(blockIdx.x), act_lds);
}

template <int MM>
static void launch_gemv(const GemmSet& g, hipStream_t st) {
    const GemmParams& p = g.p[0];
    const dim3 grid((unsigned)((p.N + 4 * kGemvCols - 1) / (4 * kGemvCols)), (unsigned)g.n);
    const size_t act_bytes = static_cast<size_t>(MM) * p.K * 2;
    const bool lds = act_bytes <= kGemvSiluLds;   // (at K of 3072 and less always)
    // Vectors of a W row in flight: what a row has, up to a whole row of 3072; loops over longer rows take half of that from
    // three activation rows on, whose products need the registers (8 rows of 3072: 33 us, 49 with whole rows).
    // us with 6 -> 3 vectors, weights in the caches: 1 x 9216 x 1536 7.5 -> 5.6, 2 rows 9.0 -> 6.9, 3 rows 10.6 -> 8.6, 4 x 6144 x 1024
    // 7.0 -> 6.2, 3 x 24576 x 4096 48.3 -> 41.5; 4 x 3072 x 12288 49.7 -> 50.6. Whole rows of 3072 beside three or four activation
    // rows pay up to 80 MiB of weights: they take 221 and 246 registers, two waves a SIMD, where half rows take 87 and 101, five
    // waves, which are worth more once a launch is many rounds of them. us with 6 -> 3, weights in the caches (from HBM): three
    // rows 12288 columns 16.9 -> 17.1 (18.4 -> 18.6), 14000 19.0 -> 18.4 (20.7 -> 19.8), 36864 45.8 -> 40.7 (45.8 -> 41.8); four rows
    // 14000 20.3 -> 20.2 (21.9 -> 21.9), 36864 48.0 -> 44.9 (48.1 -> 46.3).
    constexpr int WHOLE = MM <= 4 ? 6 : 3, LOOP = MM <= 2 ? 6 : 3;
    // The hint gains where W comes from HBM (2 to 9 %), and beside it where the activation rows are read through the cache
    // that W then leaves to them. Where the same weights are read again at once, it gains at up to 3072 of K too, but
    // costs 3 to 14 % in the loops over longer rows: us with -> without, 1 x 3072 x 12288 18.3 -> 16.1 (from HBM 20.2 -> 21.4), 3 x 18432
    // x 6144 50 -> 42 (51 -> 53). So these go without it, but for two rows, where it costs up to 5 % and gains up to 9 from HBM
    // (2 x 18432 x 6144 44.1 -> 42.1, 45.4 -> 50.1). At 3072 it loses where most of the cache is read again at once, 4 to 8 % of
    // 226 MB beside three rows and more, which gain 5 to 9 % from HBM (3 x 36864 38.4 us before these changes, 40.7 now; 45.7 and 41.8);
    // and of the activation rows that do not fit the LDS, those whose weights are more than half of the 256 MiB cache (5 x
    // 18432 x 6144 109 -> 102; 8 x 3072 x 12288 keeps it, 87.8 against 96.4).
    const int64_t w_bytes = static_cast<int64_t>(p.N) * p.K * 2 * g.n;
    const bool once = p.K <= 3072 || (lds ? MM == 2 : w_bytes <= (int64_t{128} << 20));
    const bool whole = p.K == 512 * WHOLE && (MM <= 2 || MM > 4 || w_bytes <= (int64_t{80} << 20));
#define CALL(LDS, U, EXACT, ONCE, BYTES) hipLaunchKernelGGL((gemv_small_m_kernel<MM, LDS, U, EXACT, ONCE>), grid, dim3(256), BYTES, st, g)
    if (whole) CALL(true, WHOLE, true, true, act_bytes);
    else if (p.K == 1536) CALL(true, 3, true, true, act_bytes);
    else if (p.K < 1536) CALL(true, 3, false, true, act_bytes);
    else if (lds && once) CALL(true, LOOP, false, true, act_bytes);
    else if (lds) CALL(true, LOOP, false, false, act_bytes);
    else if (once) CALL(false, LOOP, false, true, 0);
    else CALL(false, LOOP, false, false, 0);
#undef CALL
}

// ------------------------------------------------------------------------------------------------
// Any-shape kernel for operands the tiled path cannot address with 16-byte loads (K or a leading
// dimension not a multiple of 8, or a misaligned base). One thread per output element.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gemm_nt_scalar_kernel(GemmParams p) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= static_cast<int64_t>(p.M) * p.N) return;
    const int m = static_cast<int>(idx / p.N), n = static_cast<int>(idx % p.N);
    const bf16_t* a = p.A + static_cast<int64_t>(m) * p.lda;
    const bf16_t* w = p.W + static_cast<int64_t>(n) * p.ldw;
    float acc = 0.0f;
    for (int k = 0; k < p.K; ++k) {
        float x = bf2f(a[k]);
        if (p.in_silu) x = round_bf16(x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)));
        acc += x * bf2f(w[k]);
    }
    float t = acc + (p.bias ? bf2f(p.bias[n]) : 0.0f);
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

template <bool KTAIL>
static void launch_ring(const GemmSet& g, hipStream_t st) {
    const GemmLaunch L = make_launch(g, 256, 256);
    if (g.n == 1) hipLaunchKernelGGL((gemm_nt_ring_kernel<4, KTAIL, false>), dim3(grid_of(L)), dim3(kGemmThreads), 0, st, L);
    else hipLaunchKernelGGL((gemm_nt_ring_kernel<4, KTAIL, true>), dim3(grid_of(L)), dim3(kGemmThreads), 0, st, L);
}

static void launch_square(const GemmSet& g, hipStream_t st) {
    if (g.p[0].K % 64 == 0) launch_ring<false>(g, st);
    else launch_ring<true>(g, st);
}

template <int FM, int FN>
static void launch_rect(const GemmSet& g, hipStream_t st) {
    const GemmLaunch L = make_launch(g, 32 * FM, 32 * FN);
    if (g.p[0].K % 64 == 0) hipLaunchKernelGGL((gemm_nt_rect_kernel<FM, FN, false>), dim3(grid_of(L)), dim3(kGemmThreads), 0, st, L);
    else hipLaunchKernelGGL((gemm_nt_rect_kernel<FM, FN, true>), dim3(grid_of(L)), dim3(kGemmThreads), 0, st, L);
}

}  // namespace flux

using namespace flux;

// ------------------------------------------------------------------------------------------------
// Which tile for which product. The time of a launch is rounds of workgroups x (fixed + slabs x time of a
// slab), a slab being 64 of K; the constants are measured: one fit over 45 products of 100 to 13008 rows
// with 3072 to 21504 columns and K of 3072 to 15360, weights coming from HBM, every tile shape timed on
// each (largest loss of the choice against the best shape 7 %, 1 % on average; hipBLASLt through PyTorch
// in parentheses):
//   320 x 3072 x 15360   75 -> 45 us (64)       512 x 3072 x 3072    28 -> 21 us (22)
//   512 x 12288 x 3072   57 -> 43 us (43)       1280 x 3072 x 12288  141 -> 93 us (112)
//   512 x 3072 x 12288   98 -> 50 us (69)       2048 x 3072 x 3072   50 -> 40 us (40)
//   768 x 3072 x 12288   138 -> 62 us (95)      2700 x 3072 x 15360  342 -> 216 us (297)
// (before: 128-wide tiles, or 64-wide ones up to 128 tiles of 128; tiles with rows to spare excluded).
// The rectangles of 256 x 224, 224 x 256 and 224 x 288 came later, for rounds that the others leave half empty (us before
// -> now, weights from HBM; two numbers of rows share a launch):
//   4096 + 512 x 9216 x 3072   215 -> 202     1305 + 357 x 9216 x 3072   98 -> 77      1500 x 9216 x 3072    80 -> 66
//   4096 + 512 x 12288 x 3072  294 -> 278     1336 + 207 x 9216 x 3072   83 -> 71      5000 x 3072 x 3072    80 -> 71
//   4096 + 512 x 3072 x 12288  261 -> 250     876 + 138 x 12288 x 3072   85 -> 74      4702 x 3072 x 15360  317 -> 299
// A product of at least a few thousand rows fills the CUs with large tiles: one workgroup of four waves per
// CU, 256 x 256 or whichever rectangle's rounds come out shortest. Below that the eight-wave tiles, down
// to 64 x 64; what the fit shows to bound those is the load path of a CU (a slab costs in proportion to
// (FM + FN), about 50 bytes per ns), not the MFMAs, so larger tiles with K split over workgroups win
// where N alone does not give enough tiles, as long as the partial sums (written and read once, fp32)
// cost less than the rounds they save.
// ------------------------------------------------------------------------------------------------
enum TileFamily { kSquare, kRect, kPair };
struct TilePlan {
    TileFamily family;
    int fm, fn, splits;
    double us;
    bool checked = false;   // eight-wave tiles with the epilogue that decides per column
    int head_rows = 0;      // > 0: this many rows on these tiles, the rest on eight-wave ones behind them
};
struct TileShape {
    TileFamily family;
    int fm, fn;
    double slab_us;
};
static const TileShape kTileShapes[] = {
    {kSquare, 8, 8, 1.475}, {kRect, 9, 6, 1.200}, {kRect, 8, 6, 1.136}, {kRect, 7, 6, 1.042}, {kRect, 8, 7, 1.290}, {kRect, 7, 8, 1.300}, {kRect, 7, 9, 1.450},
    {kPair, 6, 6, 0.869}, {kPair, 5, 6, 0.756}, {kPair, 4, 6, 0.647}, {kPair, 8, 4, 0.838}, {kPair, 7, 4, 0.760},
    {kPair, 6, 4, 0.626}, {kPair, 5, 4, 0.568}, {kPair, 5, 3, 0.502}, {kPair, 4, 3, 0.458},
    {kPair, 3, 3, 0.325}, {kPair, 2, 3, 0.287}, {kPair, 2, 2, 0.183}, {kPair, 4, 8, 0.900},
};

static int64_t tile_count(const GemmSet& g, const TileShape& t) {
    const uint32_t bm = 32 * t.fm, bn = 32 * t.fn;   // (32-bit divisions: the search below does some forty per call)
    int64_t rows = 0;
    for (int i = 0; i < g.n; ++i) rows += (static_cast<uint32_t>(g.p[i].M) + bm - 1) / bm;
    return rows * ((static_cast<uint32_t>(g.p[0].N) + bn - 1) / bn);
}
static int64_t split_bytes(const GemmSet& g, const TileShape& t, int splits) {
    return tile_count(g, t) * splits * (32 * t.fm) * (32 * t.fn) * 4;
}

static const double kLaunch = 4.6, kTileLarge = 4.3, kTilePair = 2.7, kReduce = 1.7, kSplitGBs = 5970.0, kWeightGBs = 4500.0;
static const double kIdleShare = 0.31;   // a workgroup runs up to this much faster the emptier the GPU is
static const double kSplitHostUs = 6.0;  // K in parts costs the host this much more, ...
static const double kSplitCallUs = 20.0; // ... in all about this much

// us per slab of K. The prices were measured with weights in the Infinity Cache. From HBM a CU takes in no more than 55 bytes per ns where nobody else
// brings its weights in: one product of up to 96 rows in a single row of tiles, or, with `from_hbm`, two products of few rows (see plan_tiles).
// us, weights from HBM (from the cache), by the prices alone -> so: 64 x 3072 x 15360 44.6 -> 29.1 (27.8 -> 20.8), 90 x 3072 x 15360 37.6 -> 30.3 (24.5 ->
// 23.0), 90 x 12288 x 4096 34.5 -> 27.5 (20.7 -> 19.8), 90 x 9216 x 6144 51.0 -> 38.7 (28.8 -> 25.4). More rows: tiles of a column share its weights, and
// a single row of larger tiles is priced well enough. Bounded too, 145 x 3072 x 15360 took 33.7 (27.3) and not 37.5 (26.1), but 129 x 8192 x 8192 49.7 (37.7)
// and not 50.0 (33.4), 210 x 9216 x 6144 47.9 (36.5) and not 44.2 (34.0).
static double slab_us(const GemmSet& g, const TileShape& t, bool from_hbm) {
    const bool bound = g.n == 1 ? g.p[0].M <= std::min(96, 32 * t.fm) : from_hbm;
    return bound && weights_from_hbm(g) ? std::max(t.slab_us, (t.fm + t.fn) * 4096 / 55e3) : t.slab_us;
}

static double tile_cost_us(const GemmSet& g, const TileShape& t, int splits, bool from_hbm = false) {
    const int64_t tiles = tile_count(g, t) * splits;
    const int64_t rounds = (tiles + kGemmCUs - 1) / kGemmCUs;
    const double fill = static_cast<double>(tiles) / (rounds * kGemmCUs);
    const int slabs = ((g.p[0].K + 63) / 64 + splits - 1) / splits;
    const double us = rounds * ((t.family == kPair ? kTilePair : kTileLarge) + slabs * slab_us(g, t, from_hbm) * (1.0 - kIdleShare * (1.0 - fill)));
    // Below the time the weights take to arrive, shapes would be alike: the one with less of its own to do comes first
    // (12288 columns of 3072 at 64 rows: 64 x 64 tiles 19 us, 96 x 96 23, 192 x 128 30).
    const double weights_us = 2e-3 * g.n * g.p[0].N * g.p[0].K / kWeightGBs;
    return kLaunch + std::max(us, weights_us) + 0.05 * std::min(us, weights_us) + (splits > 1 ? kReduce + 2e-3 * split_bytes(g, t, splits) / kSplitGBs : 0.0);
}

// No more than tile_cost_us in `splits` or more parts: the work spread evenly over the CUs, and the traffic of the parts.
static double split_floor_us(const GemmSet& g, const TileShape& t, int splits, bool from_hbm) {
    return kLaunch + kReduce + kTilePair + tile_count(g, t) * (g.p[0].K / 64) * slab_us(g, t, from_hbm) / kGemmCUs + 2e-3 * split_bytes(g, t, splits) / kSplitGBs;
}

// The best eight-wave tile for a product whose K is not cut.
static TilePlan plan_eight_waves(const GemmSet& g) {
    TilePlan best = {kPair, 0, 0, 1, 1e30, true};
    for (const TileShape& t : kTileShapes) {
        if (t.family != kPair || t.fn == 8) continue;
        const double us = tile_cost_us(g, t, 1);
        if (us < best.us) best = {kPair, t.fm, t.fn, 1, us, true};
    }
    return best;
}

// The first `rows` rows of a product, or those behind them.
static GemmSet rows_before(const GemmSet& g, int rows) {
    GemmSet head = g;
    head.p[0].M = rows;
    return head;
}
static GemmSet rows_behind(const GemmSet& g, int rows) {
    GemmSet tail = g;
    GemmParams& t = tail.p[0];
    const int64_t row0 = rows;
    t.M -= rows;
    t.A += row0 * t.lda;
    t.Y += row0 * t.ldy;
    if (t.Y2 != nullptr) t.Y2 += row0 * t.ldy2;
    if (t.gate != nullptr) {
        t.resid += row0 * t.ldresid;
        t.gate += row0 / t.rows_per_batch * t.gate_stride;
    }
    return tail;
}

static TilePlan plan_priced(const GemmSet& g, bool shared_gpu, int64_t workspace_bytes, bool from_hbm) {
    // The branch-free epilogue of the rectangular and eight-wave tiles: 16-byte outputs, a wave's columns on one
    // side of split_n and act_begin, no GELU in front of a gate. The square and the eight-wave tiles have one for
    // anything else as well. (Without it on the eight-wave tiles, calls outside the form ran on square ones: 64 x 3072
    // x 3072 with 1000 columns in the first output 13 -> 63 us, 300 x 1001 x 3072 14 -> 30 us.)
    const GemmParams& p = g.p[0];
    // near288: also 288 rows of W lie within 32-bit byte offsets, as 256 of them do on every call that gets here. Past
    // that, offsets reach kOutOfRange and the K tail of those rows is no longer read as zeros.
    bool form = true, near288 = true;
    for (int i = 0; i < g.n; ++i) {
        const GemmParams& q = g.p[i];
        near288 = near288 && q.ldw * 2 * 288 < 0x7fffffffLL;
        form = form && q.vec_io && q.N % 8 == 0 && (q.bias == nullptr || q.bias_vec) && !(q.gate != nullptr && q.act != FLUX_ACT_NONE) &&
               q.lda * 2 * 288 < 0x7fffffffLL && q.ldw * 2 * 256 < 0x7fffffffLL && q.ldy * 2 * 288 < 0x7fffffffLL &&
               q.ldy2 * 2 * 288 < 0x7fffffffLL && q.ldresid * 2 * 288 < 0x7fffffffLL;   // 32-bit byte offsets inside a tile's rows
    }
    auto columns_ok = [&](int fn) {
        const int w = 16 * fn;
        return form && (fn <= 8 || near288) && (p.split_n >= p.N || p.split_n % w == 0) && (p.act == FLUX_ACT_NONE || p.act_begin >= p.N || p.act_begin % w == 0);
    };
    if (!form && p.qk_cols > 0) return {kSquare, 8, 8, 1, 0.0};   // (whole heads per wave: 256-wide tiles only)
    TilePlan best = {kSquare, 8, 8, 1, 1e30};
    // Calls with the q/k epilogue take the cheapest shape whose waves hold whole heads (128 columns), whatever the plain
    // product of that size takes. Fused projection of the single block (21504 x 3072, weights from HBM), us on 256 x
    // 256, 224 x 256 and eight-wave 128 x 256 tiles: 320 rows 79 75 58, 640 88 79 108, 1153 159 142 173, 1920 243 215
    // 256, 2049 237 263 290, 3329 409 367 424, 4608 492 517 560. (The eight-wave tile sums K in another order.)
    for (const TileShape& t : kTileShapes) {
        if (p.qk_cols > 0 ? t.fn != 8 : t.fn == 8 && t.family == kPair) continue;   // (eight waves of that width are there for q/k only)
        // Rectangles of 50000 outputs and more: measured from K = 1024 on. Their epilogues, which a slab's price does not
        // hold, are as long as the square tile's. Beside another stream no rectangle is taken in the end (below), and these,
        // which replace eight-wave tiles too, would only hide those: 6100 x 9216 x 3072 272 us, 292 on square tiles.
        if (t.family == kRect && t.fn > 6 && p.qk_cols == 0 && (p.K < 1024 || shared_gpu)) continue;
        if ((t.family == kRect || (t.family == kPair && t.fn == 8)) && !columns_ok(t.fn)) continue;
        const double us = tile_cost_us(g, t, 1, from_hbm);
        if (us < best.us) best = {t.family, t.fm, t.fn, 1, us, t.family == kPair && !columns_ok(t.fn)};
    }
    // K in parts, where that gains more than the host pays for it: a workspace to allocate and a second launch, 6 us
    // per call (64 x 3072 x 3072 takes 11 us of the GPU in two parts and 13 in one, but the host 20 and 14), and where
    // the product in one piece takes the GPU longer than the call in parts takes the host.
    if (workspace_bytes > 0 && best.us > kSplitCallUs && p.K % 64 == 0 && p.K / 64 >= 8 && p.qk_cols == 0) {
        const double bar = best.us - kSplitHostUs;
        TilePlan split = {kPair, 0, 0, 1, bar};
        for (const TileShape& t : kTileShapes) {
            if (t.family != kPair || t.fn == 8) continue;
            for (int s = 2; s <= 10; ++s) {
                if (tile_count(g, t) * s > 2 * kGemmCUs || (p.K / 64) / s < 4 || split_bytes(g, t, s) > workspace_bytes) break;
                if (split_floor_us(g, t, s, from_hbm) > split.us) break;
                const double us = tile_cost_us(g, t, s, from_hbm);
                if (us < split.us) split = {kPair, t.fm, t.fn, s, us, !columns_ok(t.fn)};
            }
        }
        if (split.splits > 1) best = split;
    }
    // Where rectangles may be missing (192 columns are whole waves of every tile): whole rounds of 256-wide tiles
    // with the rows left over on eight-wave ones behind them, instead of a last round that is mostly empty.
    // Only along the edge of a batch element, whose gate vector a part starts with.
    const int64_t tiles = tile_count(g, kTileShapes[0]), tiles_n = (p.N + 255) / 256;
    if (!columns_ok(12) && p.qk_cols == 0 && g.n == 1 && p.a_skip == 0 && tiles > kGemmCUs) {
        const int64_t most = tiles / kGemmCUs * kGemmCUs / tiles_n;   // tile rows in whole rounds
        for (int64_t c = most; c > 0 && c > most - 4; --c) {
            const int rows = static_cast<int>(c * 256);
            if (rows >= p.M || (p.gate != nullptr && rows % p.rows_per_batch != 0)) continue;
            const double us = tile_cost_us(rows_before(g, rows), kTileShapes[0], 1) + plan_eight_waves(rows_behind(g, rows)).us;
            if (us < best.us) best = {kSquare, 8, 8, 1, us, false, rows};
        }
    }
    // Beside another stream's work: square tiles leave that work the CUs of their last round.
    if (shared_gpu && best.family == kRect) best = {kSquare, 8, 8, 1, best.us};
    return best;
}

// Two products of few rows share few columns of weights among their tiles, so what HBM feeds a CU bounds them as well, where the weights come from
// there. A plan is then made both ways, and the one by that bound is taken where it gains at least 3.5 us by it: smaller gains are within what the
// model is off by (258 + 498 x 6144 x 6144 72 us by the prices, 81 by the bound, for 1.4 us less in the model; 312 + 35 x 3072 x 12288 49 and 51 for 3.0,
// 168 + 488 x 9216 x 3072 48 and 53 for 1.2). Up to 768 rows and K = 12288: beyond, either plan may be the worse one (1536 + 256 x 3072 x 12288 136 us by the
// prices and 147 by the bound, 713 + 279 x 16384 x 4096 142 and 158, 150 + 10 x 4096 x 16384 70 and 78).
// us, weights from HBM (from the cache), by the prices -> so: 256 + 64 x 3072 x 12288 67.3 -> 48.5 (42.3 -> 38.1), 80 + 40 58.0 -> 43.6 (39.9 -> 30.6), 570 +
// 20 88.4 -> 63.5 (59.7 -> 55.1), 660 + 60 86.0 -> 70.4 (60.1 -> 65.3), 89 + 272 58.2 -> 49.7 (38.9 -> 41.5), 113 + 53 x 9216 x 3072 37.8 -> 33.5 (25.7 -> 23.7).
static TilePlan plan_tiles(const GemmSet& g, bool shared_gpu, int64_t workspace_bytes) {
    const TilePlan plan = plan_priced(g, shared_gpu, workspace_bytes, false);
    if (g.n == 1 || g.p[0].M + g.p[1].M > 768 || g.p[0].K > 12288 || !weights_from_hbm(g)) return plan;
    const TilePlan bound = plan_priced(g, shared_gpu, workspace_bytes, true);
    auto cost = [&](const TilePlan& of) {
        for (const TileShape& t : kTileShapes)
            if (t.family == of.family && t.fm == of.fm && t.fn == of.fn) return tile_cost_us(g, t, of.splits, true);
        return 0.0;
    };
    return cost(plan) - cost(bound) >= 3.5 ? bound : plan;
}

// How a call can be served.
enum LinearRoute { kNothing, kScalar, kRows, kTiles };

// Checks a call and turns it into the kernels' parameters.
static int read_linear_args(const flux_linear_args* a, GemmParams& p, LinearRoute& route) {
    route = kNothing;
    if (!a) return fail(FLUX_E_NULL, "flux_linear_bf16: null args");
    if (!a->A || !a->W || !a->Y) return fail(FLUX_E_NULL, "flux_linear_bf16: null operand");
    if (a->M < 0 || a->N < 0 || a->K < 0) return fail(FLUX_E_SHAPE, "flux_linear_bf16: negative size");
    if (a->M > 0x7fffffff || a->N > 0x7fffffff || a->K > 0x7fffffff) return fail(FLUX_E_SHAPE, "flux_linear_bf16: size exceeds 2^31");
    if (a->M == 0 || a->N == 0) return FLUX_OK;
    if (a->lda < a->K || a->ldw < a->K) return fail(FLUX_E_SHAPE, "flux_linear_bf16: leading dimension smaller than K");
    if (a->act != FLUX_ACT_NONE && a->act != FLUX_ACT_GELU_TANH) return fail(FLUX_E_UNSUPPORTED, "flux_linear_bf16: unknown activation %d", a->act);
    if ((a->flags & ~static_cast<int64_t>(FLUX_LINEAR_SHARED_GPU)) != 0) return fail(FLUX_E_UNSUPPORTED, "flux_linear_bf16: unknown flags 0x%llx", (unsigned long long)a->flags);
    if (a->in_act != FLUX_ACT_NONE && a->in_act != FLUX_ACT_SILU) return fail(FLUX_E_UNSUPPORTED, "flux_linear_bf16: unknown input activation %d", a->in_act);
    if (a->in_act == FLUX_ACT_SILU && (a->M > 8 || a->qk != nullptr)) return fail(FLUX_E_UNSUPPORTED, "flux_linear_bf16: input SiLU is for M <= 8 without the qk fusion (M=%lld)", (long long)a->M);
    const bool split = a->Y2 != nullptr && a->split_n < a->N;
    if (split && (a->split_n < 0 || a->y2_col0 < 0)) return fail(FLUX_E_SHAPE, "flux_linear_bf16: bad split");
    if ((a->gate == nullptr) != (a->resid == nullptr)) return fail(FLUX_E_NULL, "flux_linear_bf16: gate and resid go together");
    if (a->gate && a->rows_per_batch <= 0) return fail(FLUX_E_SHAPE, "flux_linear_bf16: rows_per_batch must be positive with a gate");

    p.A = static_cast<const bf16_t*>(a->A); p.W = static_cast<const bf16_t*>(a->W); p.bias = static_cast<const bf16_t*>(a->bias);
    p.Y = static_cast<bf16_t*>(a->Y); p.Y2 = split ? static_cast<bf16_t*>(a->Y2) : nullptr;
    p.resid = static_cast<const bf16_t*>(a->resid); p.gate = static_cast<const bf16_t*>(a->gate);
    p.M = (int)a->M; p.N = (int)a->N; p.K = (int)a->K;
    p.a_rows = 1; p.a_skip = 0;
    p.lda = a->lda; p.ldw = a->ldw; p.ldy = a->ldy; p.ldy2 = a->ldy2; p.ldresid = a->ldresid;
    p.gate_stride = a->gate_batch_stride;
    p.split_n = split ? (int)a->split_n : p.N;
    p.y2_col0 = split ? (int)a->y2_col0 : 0;
    p.rows_per_batch = a->gate ? (int)a->rows_per_batch : 1;
    p.in_silu = a->in_act == FLUX_ACT_SILU;
    p.checked = 0;
    p.act = a->act; p.act_begin = (int)(a->act_begin < 0 ? 0 : (a->act_begin > a->N ? a->N : a->act_begin));
    p.bias_vec = a->bias != nullptr && (reinterpret_cast<uintptr_t>(a->bias) & 3u) == 0 && a->N % 4 == 0;
    p.vec_io = aligned16(a->Y) && a->ldy % 8 == 0 &&
               (!split || (aligned16(a->Y2) && a->ldy2 % 8 == 0 && a->split_n % 8 == 0 && a->y2_col0 % 8 == 0)) &&
               (!a->gate || (aligned16(a->gate) && aligned16(a->resid) && a->ldresid % 8 == 0 && a->gate_batch_stride % 8 == 0));

    p.q_out = p.k_out = nullptr; p.q_scale = p.k_scale = nullptr; p.pe = nullptr; p.pe_batch_stride = 0;
    p.qk_cols = p.qk_heads = p.qk_seq_len = p.qk_out_len = p.qk_pos0 = 0; p.qk_eps = 0.0f;
    if (a->qk != nullptr) {
        const flux_linear_qk_fusion* f = a->qk;
        if (!f->q_out || !f->k_out || !f->q_scale || !f->k_scale || !f->pe) return fail(FLUX_E_NULL, "flux_linear_bf16: qk fusion with a null pointer");
        const int64_t cols = 2 * f->heads * 128;
        const bool shape_ok = f->heads > 0 && f->seq_len >= 256 && a->M % f->seq_len == 0 && a->N % 256 == 0 &&
                              cols <= a->N && f->pos0 >= 0 && f->pos0 + f->seq_len <= f->out_len && f->out_len < 0x7fffff &&
                              f->heads * f->out_len * 256 < 0x7fffffffLL &&
                              f->pe_batch_stride >= 0 && a->K > 0 && a->K % 8 == 0;
        const bool epi_ok = a->gate == nullptr && p.act_begin >= cols && p.split_n >= cols &&
                            (a->bias == nullptr || p.bias_vec) && p.vec_io;
        const bool ptr_ok = aligned16(f->q_out) && aligned16(f->k_out) && aligned16(f->pe) && f->pe_batch_stride % 4 == 0 &&
                            (reinterpret_cast<uintptr_t>(f->q_scale) & 3u) == 0 && (reinterpret_cast<uintptr_t>(f->k_scale) & 3u) == 0 &&
                            aligned16(a->A) && aligned16(a->W) && a->lda % 8 == 0 && a->ldw % 8 == 0 &&
                            a->lda * 2 * 256 < 0x7fffffffLL && a->ldw * 2 * 256 < 0x7fffffffLL;
        if (!shape_ok || !epi_ok || !ptr_ok)
            return fail(FLUX_E_UNSUPPORTED, "flux_linear_bf16: qk fusion needs N in multiples of 256, sequences of at least 256 rows, "
                                            "aligned operands, no gate, and GELU / split columns behind the k heads");
        p.q_out = static_cast<bf16_t*>(f->q_out); p.k_out = static_cast<bf16_t*>(f->k_out);
        p.q_scale = static_cast<const bf16_t*>(f->q_scale); p.k_scale = static_cast<const bf16_t*>(f->k_scale);
        p.pe = f->pe; p.pe_batch_stride = f->pe_batch_stride;
        p.qk_cols = (int)cols; p.qk_heads = (int)f->heads; p.qk_seq_len = (int)f->seq_len; p.qk_out_len = (int)f->out_len;
        p.qk_pos0 = (int)f->pos0; p.qk_eps = f->eps;
    }
    const bool vec_in = aligned16(a->A) && aligned16(a->W) && a->K % 8 == 0 && a->lda % 8 == 0 && a->ldw % 8 == 0;
    // 32-bit byte offsets inside one tile's rows
    const bool off_ok = a->lda * 2 * 256 < 0x7fffffffLL && a->ldw * 2 * 256 < 0x7fffffffLL;
    // (degenerate contraction, K = 0: the scalar kernel's empty K loop leaves bias and epilogue only)
    route = p.K == 0 || !vec_in || !off_ok ? kScalar : (p.M <= 8 && p.qk_cols == 0 ? kRows : kTiles);
    return FLUX_OK;
}

static int launch_rows(const GemmSet& g, hipStream_t st) {
    switch (g.p[0].M) {
        case 1: launch_gemv<1>(g, st); break;
        case 2: launch_gemv<2>(g, st); break;
        case 3: launch_gemv<3>(g, st); break;
        case 4: launch_gemv<4>(g, st); break;
        case 5: launch_gemv<5>(g, st); break;
        case 6: launch_gemv<6>(g, st); break;
        case 7: launch_gemv<7>(g, st); break;
        default: launch_gemv<8>(g, st); break;
    }
    return check_launch("flux_linear_bf16");
}

// With `need` nothing is launched: it receives the workspace the launch would like to have.
static int launch_tiles(GemmSet& g, bool shared_gpu, void* workspace, int64_t workspace_bytes, int64_t* need, hipStream_t st) {
    const TilePlan plan = plan_tiles(g, shared_gpu, need != nullptr ? INT64_MAX : workspace_bytes);
    if (need != nullptr) {
        if (plan.splits > 1) *need = split_bytes(g, {plan.family, plan.fm, plan.fn, 0.0}, plan.splits);
        return FLUX_OK;
    }
    if (plan.head_rows > 0) {
        GemmSet tail = rows_behind(g, plan.head_rows);
        const TilePlan behind = plan_eight_waves(tail);
        tail.p[0].checked = 1;
        launch_square(rows_before(g, plan.head_rows), st);
        launch_pair_tiles(behind.fm, behind.fn, tail, 1, nullptr, st);
        return check_launch("flux_linear_bf16");
    }
    for (int i = 0; i < g.n; ++i) g.p[i].checked = plan.checked;
    switch (plan.family) {
        case kSquare: launch_square(g, st); break;
        case kRect:
            if (plan.fm == 9) launch_rect<9, 6>(g, st);
            else if (plan.fm == 8 && plan.fn == 7) launch_rect<8, 7>(g, st);
            else if (plan.fm == 8) launch_rect<8, 6>(g, st);
            else if (plan.fn == 9) launch_rect<7, 9>(g, st);
            else if (plan.fn == 6) launch_rect<7, 6>(g, st);
            else launch_rect<7, 8>(g, st);
            break;
        case kPair: launch_pair_tiles(plan.fm, plan.fn, g, plan.splits, static_cast<float*>(workspace), st); break;
    }
    return check_launch("flux_linear_bf16");
}

static int linear_launch(const flux_linear_args* a, void* workspace, int64_t workspace_bytes, int64_t* need, hipStream_t st) {
    GemmSet g;
    LinearRoute route;
    g.n = 1;
    const int rc = read_linear_args(a, g.p[0], route);
    if (rc != FLUX_OK || route == kNothing) return rc;
    if (route == kTiles) return launch_tiles(g, (a->flags & FLUX_LINEAR_SHARED_GPU) != 0, workspace, workspace_bytes, need, st);
    if (need != nullptr) return FLUX_OK;
    if (route == kRows) { g.p[1] = g.p[0]; return launch_rows(g, st); }
    const GemmParams& p = g.p[0];
    hipLaunchKernelGGL(gemm_nt_scalar_kernel, dim3((unsigned)(((int64_t)p.M * p.N + 255) / 256)), dim3(256), 0, st, p);
    return check_launch("flux_linear_bf16");
}

// Rows of A in batches whose distance is not rows x lda (a slice of a longer sequence).
static int set_a_batches(GemmParams& p, int64_t rows, int64_t stride, LinearRoute route, const char* what) {
    if (rows == 0) return FLUX_OK;
    if (rows < 0 || stride < 0) return fail(FLUX_E_SHAPE, "%s: negative rows or stride of A's batches", what);
    if (route == kNothing || p.M <= rows || stride == rows * p.lda) return FLUX_OK;
    if (route != kTiles || stride % 8 != 0 || stride < rows * p.lda || ((p.M - 1) / rows + 1) * stride * 2 >= 0x7fffffffLL)
        return fail(FLUX_E_UNSUPPORTED, "%s: batches of A need more than 8 rows in all, a stride of a multiple of 8 and less than 2 GiB in all", what);
    p.a_rows = (int)rows;
    p.a_skip = stride - rows * p.lda;
    return FLUX_OK;
}

static bool share_launch(const GemmSet& g, const LinearRoute (&route)[2]) {
    const GemmParams &p = g.p[0], &q = g.p[1];
    const bool same = route[0] == route[1] && p.N == q.N && p.K == q.K && p.act == q.act && p.act_begin == q.act_begin && p.split_n == q.split_n &&
                      p.in_silu == q.in_silu && (p.gate != nullptr) == (q.gate != nullptr) && p.qk_cols == q.qk_cols;
    return same && (route[0] == kTiles || (route[0] == kRows && p.M == q.M));
}

// One launch for both products where they have the same N, K and form of epilogue, so that the tile grid is
// that of their rows together; else one after the other through the same workspace (the stream orders them).
// 1024 + 256 rows of the double-stream block, one launch against two on two streams: 3072 x 9216 weights 59 us
// (55 and 31 side by side), 12288 x 3072 81 (66, 33), 3072 x 12288 101 (85, 36); the pass 567 -> 371 us.
static int linear_pair_launch(const flux_linear_pair_args* a, void* workspace, int64_t workspace_bytes, int64_t* need, hipStream_t st) {
    if (!a) return fail(FLUX_E_NULL, "flux_linear_bf16_pair: null args");
    GemmSet g;
    LinearRoute route[2];
    for (int i = 0; i < 2; ++i) {
        int rc = read_linear_args(&a->product[i], g.p[i], route[i]);
        if (rc == FLUX_OK) rc = set_a_batches(g.p[i], a->a_rows[i], a->a_batch_stride[i], route[i], "flux_linear_bf16_pair");
        if (rc != FLUX_OK) return rc;
    }
    const bool shared_gpu = ((a->product[0].flags | a->product[1].flags) & FLUX_LINEAR_SHARED_GPU) != 0;
    if (need != nullptr) *need = 0;
    if (share_launch(g, route)) {
        g.n = 2;
        if (route[0] == kTiles) return launch_tiles(g, shared_gpu, workspace, workspace_bytes, need, st);
        return need != nullptr ? FLUX_OK : launch_rows(g, st);
    }
    for (int i = 0; i < 2; ++i) {
        int64_t part = 0;
        int rc;
        if (route[i] == kTiles) {
            GemmSet one;
            one.n = 1;
            one.p[0] = g.p[i];
            rc = launch_tiles(one, shared_gpu, workspace, workspace_bytes, need != nullptr ? &part : nullptr, st);
        } else {
            rc = linear_launch(&a->product[i], workspace, workspace_bytes, need != nullptr ? &part : nullptr, st);
        }
        if (rc != FLUX_OK) return rc;
        if (need != nullptr) *need = std::max(*need, part);
    }
    return FLUX_OK;
}

namespace flux {
bool rows_beside(const flux_linear_pair_args* a, GemmSet& g, int& rc) {
    LinearRoute route[2];
    rc = FLUX_OK;
    for (int i = 0; i < 2 && rc == FLUX_OK; ++i) {
        rc = read_linear_args(&a->product[i], g.p[i], route[i]);
        if (rc == FLUX_OK) rc = set_a_batches(g.p[i], a->a_rows[i], a->a_batch_stride[i], route[i], "flux_attention_rows_bf16");
    }
    if (rc != FLUX_OK || route[0] != kRows) return false;
    g.n = route[1] == kNothing ? 1 : 2;
    if (g.n == 1) g.p[1] = g.p[0];
    return g.n == 1 || share_launch(g, route);
}
}  // namespace flux

extern "C" int flux_linear_bf16(const flux_linear_args* a, void* stream) {
    return linear_launch(a, nullptr, 0, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int64_t flux_linear_workspace_bytes(const flux_linear_args* a) {
    int64_t need = 0;
    return linear_launch(a, nullptr, 0, &need, nullptr) == FLUX_OK ? need : 0;
}

extern "C" int flux_linear_bf16_ws(const flux_linear_args* a, void* workspace, int64_t workspace_bytes, void* stream) {
    if (workspace_bytes < 0 || (workspace_bytes > 0 && (!workspace || !aligned16(workspace)))) return fail(FLUX_E_NULL, "flux_linear_bf16_ws: workspace must be 16-byte aligned memory");
    return linear_launch(a, workspace, workspace_bytes, nullptr, static_cast<hipStream_t>(stream));
}

extern "C" int64_t flux_linear_pair_workspace_bytes(const flux_linear_pair_args* a) {
    int64_t need = 0;
    return linear_pair_launch(a, nullptr, 0, &need, nullptr) == FLUX_OK ? need : 0;
}

extern "C" int flux_linear_bf16_pair(const flux_linear_pair_args* a, void* workspace, int64_t workspace_bytes, void* stream) {
    if (workspace_bytes < 0 || (workspace_bytes > 0 && (!workspace || !aligned16(workspace)))) return fail(FLUX_E_NULL, "flux_linear_bf16_pair: workspace must be 16-byte aligned memory");
    return linear_pair_launch(a, workspace, workspace_bytes, nullptr, static_cast<hipStream_t>(stream));
}

// The q/k epilogue needs waves of 128 columns, which leaves three tile shapes. Where those need a round that is mostly empty, or twice the rows,
// a plain product on a better shape and the preparation kernel behind it take less. Both are priced here: the product as plan_tiles does,
// the epilogue 1.5 us on eight-wave tiles and 5 on the others, the preparation 4.2 us of launch and latency and 0.83 us per million values of q
// and k, fitted to passes of the single block of 24 heads and 21504 columns. Passes with the epilogue and with the preparation (us): 320 rows 127.4
// and 124.1, 384 134.7 135.2, 448 157.5 144.3, 512 161.4 153.2, 640 176.0 178.0, 704 196.0 205.3, 896 258.0 242.3, 1024 272.1 261.6, 1280 303.7
// 307.4. From three rounds on the prices are off by as much as the two differ: 1700 414.2 and 424.2, priced 2.5 the other way.
extern "C" int flux_linear_qk_pays(int64_t M, int64_t N, int64_t K, int64_t heads) {
    if (M <= 0 || N <= 0 || K <= 0 || heads <= 0 || M > INT_MAX || N > INT_MAX || K > INT_MAX || heads > N / 256) return 1;
    GemmSet g = {};
    g.n = 1;
    GemmParams& p = g.p[0];
    p.M = static_cast<int>(M);
    p.N = static_cast<int>(N);
    p.K = static_cast<int>(K);
    p.lda = p.ldw = K;
    p.ldy = p.ldy2 = N;
    p.rows_per_batch = p.M;
    p.split_n = p.act_begin = static_cast<int>(std::min(N, 3 * heads * 128));
    p.act = FLUX_ACT_GELU_TANH;
    p.vec_io = 1;
    const TilePlan plain = plan_tiles(g, false, 0);
    p.qk_cols = static_cast<int>(2 * heads * 128);
    const TilePlan fused = plan_tiles(g, false, 0);
    if (tile_count(g, {fused.family, fused.fm, fused.fn, 0.0}) > 2 * kGemmCUs) return 1;
    const double prepared = 4.2 + 0.83e-6 * static_cast<double>(M) * p.qk_cols;
    return fused.us + (fused.family == kPair ? 1.5 : 5.0) <= plain.us + prepared ? 1 : 0;
}

extern "C" int flux_linear_plan_of(const flux_linear_args* first, const flux_linear_args* second, int64_t workspace_bytes, flux_linear_plan* plan) {
    if (!plan) return fail(FLUX_E_NULL, "flux_linear_plan_of: null plan");
    *plan = {FLUX_LINEAR_NOTHING, 0, 0, 1, 1, 0, 0};
    GemmSet g;
    LinearRoute route[2];
    int rc = read_linear_args(first, g.p[0], route[0]);
    if (rc == FLUX_OK && second) rc = read_linear_args(second, g.p[1], route[1]);
    if (rc != FLUX_OK) return rc;
    plan->products = g.n = second && share_launch(g, route) ? 2 : 1;
    if (route[0] == kScalar) plan->family = FLUX_LINEAR_SCALAR;
    if (route[0] == kRows) plan->family = FLUX_LINEAR_ROWS;
    if (route[0] != kTiles) return FLUX_OK;
    const bool shared_gpu = ((first->flags | (g.n > 1 ? second->flags : 0)) & FLUX_LINEAR_SHARED_GPU) != 0;
    const TilePlan t = plan_tiles(g, shared_gpu, workspace_bytes);
    plan->family = t.family == kSquare ? FLUX_LINEAR_SQUARE : t.family == kRect ? FLUX_LINEAR_RECT : FLUX_LINEAR_EIGHT_WAVES;
    plan->tile_m = 32 * t.fm;
    plan->tile_n = 32 * t.fn;
    plan->splits = t.splits;
    plan->head_rows = t.head_rows;
    plan->checked = t.checked || t.family == kSquare;
    return FLUX_OK;
}
