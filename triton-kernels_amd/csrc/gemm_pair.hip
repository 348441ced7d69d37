// Linear layer on the matrix cores, middle sizes: a few hundred to a few thousand rows.
#include "gemm_common.h"

#include <climits>

namespace flux {

// ------------------------------------------------------------------------------------------------
// Middle sizes: eight waves on a (32*FM) x (32*FN) tile, two per SIMD, as two groups of four. Both groups
// hold accumulators of the whole tile; of every K = 64 slab group 0 multiplies the first K = 32 step and
// group 1 the second, and the two sums are added through LDS at the end. A single wave per SIMD issues in
// order, and on tiles that are small enough for a few hundred rows its fragment reads (18 cycles each) and
// LDS-writing loads (34 to 64) take longer than its MFMAs; two waves that share the slab, and with it the
// LDS traffic, fill each other's gaps. ST slabs of LDS, round-robin: fragments of slab kt + 1 are read
// while slab kt is multiplied, so behind the barrier of slab kt its buffer takes slab kt + ST, and
// ST - 1 slabs are in flight or waiting.
// What bounds it: the bytes a CU can have in flight. With everything but the loads taken out 320 x 21504 x
// 3072 (160 x 192 tiles) takes 50 us with W coming from HBM and 32 us from the Infinity Cache, 50 and 38 us
// as it is, 30 us with neither loads nor fragment reads; a CU's loads stop at about 55 bytes per ns from HBM and
// 104 from the caches however many slabs are in flight. So the tile shape is chosen for few bytes per
// product. Measured (weights from HBM, before -> now): 320 x 3072 x 15360 75 -> 45 us, 768 x 3072 x 12288
// 138 -> 62 us, 1280 x 3072 x 12288 141 -> 93 us, 512 x 3072 x 3072 28 -> 21 us; a four-wave workgroup on the
// same tiles: 50, 78, 120 and 21 us.
// ------------------------------------------------------------------------------------------------
// Slabs out of turn. Tiles that share columns of W run side by side and ask for the same slab at the same time, so each of them waits for it to
// come from HBM. Where W is too large to be found in the Infinity Cache, the tiles of a column take every two or four slabs of K (`turns`, as many as there
// are tiles, or one more than three) in an order of their own, slab i ^ turn: each is the first at some of a group and finds the others in the L2, where its
// neighbours have brought them. The same goes for A among the tiles of a row. us, W from HBM, in turn -> so: 320 x 21504 x 3072 50.4 -> 47.3, 320 x 3072 x
// 15360 45.2 -> 44.5, 640 65.7 -> 63.9, 1024 101.7 -> 92.3, 1600 154.9 -> 135.4, 1900 169.3 -> 154.4, 2048 177.4 -> 158.5. A W of more than a third of
// that cache that is found there all the same costs 40.0 -> 40.4, 39.9 -> 40.5, 60.0 -> 61.6, 86.9 -> 89.4, 126.8 -> 127.9, 145.1 -> 148.4 and 150.2 -> 153.7 us; a smaller one is walked in turn.
// The order has to be cheap: rotated by additions, a branch at the end of a group and a division at the head of the kernel, all tiles in turn took 3 % longer at 1600 and 1900
// rows (130.6 and 148.9 us from the cache; 139.5 and 159.2 rotated, from HBM), and inside a slab instead of between two the order took 1 % of 512 x 3072 x 3072.
// Two products in a launch gain nothing (1024 + 256 x 3072 x 12288 99.6 and 100.2): the second's one row of tiles has nobody to share with and ends
// last. Groups of two and four times as many slabs: 48.0 and 49.2 us at the first size, 46.8 so. From four tile rows on the last one has to be three quarters full: one of
// mostly padding runs ahead of its neighbours and is then the first at every slab (K = 15360, hardly filled: 1152 rows 102.8 -> 106.1, 1402 118.4 -> 121.1, 1750
// 149.0 -> 154.2, 2100 170.8 -> 175.6, in turn now).
constexpr int kPairThreads = 512;

template <int FM, int FN, int ST, bool KTAIL, int G>
__device__ __forceinline__ void gemm_pair_slabs(const GemmParams& p, char* lds, int m0, int n0, int kb, int ke, int turn, int turns, int w4, int lane, f32x4 (&acc)[FM][FN]) {
    constexpr int BM = 32 * FM, BN = 32 * FN, BK = 64, ROWB = BK * 2;
    constexpr int SLAB = (BM + BN) * ROWB;       // A rows, then W rows
    constexpr int NL = (FM + FN + 1 - G) / 2;    // loads of this wave per slab: passes of 32 rows, every other one
    constexpr int WROWS = 16 * FM, WCOLS = 16 * FN;
    constexpr int READS = FM + FN, MFMAS = FM * FN;
    constexpr int BS = READS / 4;                // slots in front of the barrier
    static_assert(2 * (READS - BS) >= READS && READS - BS >= NL && MFMAS >= READS, "schedule shape");
    static_assert(ST >= 3 && (ST - 1) * NL <= 63 && ST * SLAB <= 160 * 1024, "ring shape");
    const int wm = w4 >> 1, wn = w4 & 1;

    const int lrow = w4 * 8 + (lane >> 3);
    const int lchunk = (lane & 7) ^ ((lrow >> 1) & 7);
    const int rows_a = min(p.M - m0, BM), rows_b = min(p.N - n0, BN);
    const int64_t a0 = row_of_a(p, m0);
    bf16_t* const base_a = const_cast<bf16_t*>(p.A + a0);
    bf16_t* const base_b = const_cast<bf16_t*>(p.W + static_cast<int64_t>(n0) * p.ldw);
    const int bytes_a = static_cast<int>((row_of_a(p, m0 + rows_a - 1) - a0 + p.K) * 2);
    const int bytes_b = static_cast<int>(((rows_b - 1) * p.ldw + p.K) * 2);
    uint32_t voff[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const int pass = 2 * j + G;
        if (pass < FM) {
            const int r = pass * 32 + lrow;
            voff[j] = r < rows_a ? static_cast<uint32_t>((row_of_a(p, m0 + r) - a0 + lchunk * 8) * 2) : kOutOfRange;
        } else {
            const int r = (pass - FM) * 32 + lrow;
            voff[j] = r < rows_b ? static_cast<uint32_t>((r * p.ldw + lchunk * 8) * 2) : kOutOfRange;
        }
    }
    // slabs from ke on read as zeros, which keeps the number of loads in flight the same to the last slab
    auto load = [&](int soff, int j, int kt) {
        const int pass = 2 * j + G;
        const bool in = kt < ke;
        const uint32_t v = KTAIL && kt * BK + lchunk * 8 >= p.K ? kOutOfRange : voff[j];
        if (pass < FM) load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_a, 0, in ? bytes_a : 0, kRsrcFlags), lds + soff + pass * 4096 + w4 * 1024, v, kt * ROWB);
        else load_chunk(__builtin_amdgcn_make_buffer_rsrc(base_b, 0, in ? bytes_b : 0, kRsrcFlags), lds + soff + pass * 4096 + w4 * 1024, v, kt * ROWB);
    };

    const int frow = lane & 15, fq = lane >> 4;
    const int ko = ((G * 4 + fq) ^ ((frow >> 1) & 7)) * 16;
    const int koff_a = (wm * WROWS + frow) * ROWB + ko;
    const int koff_w = BM * ROWB + (wn * WCOLS + frow) * ROWB + ko;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

    bf16x8 xa[2][FM], wb[2][FN];
    auto read_frag = [&](int buf, int soff, int r) {
        if (r == 0) xa[buf][0] = *reinterpret_cast<const bf16x8*>(lds + (soff + koff_a));
        else if (r <= FN) wb[buf][r - 1] = *reinterpret_cast<const bf16x8*>(lds + (soff + koff_w) + (r - 1) * 16 * ROWB);
        else xa[buf][r - FN] = *reinterpret_cast<const bf16x8*>(lds + (soff + koff_a) + (r - FN) * 16 * ROWB);
    };
    auto mfma_one = [&](int buf, int idx) {
        const int i = idx / FN, j = (i & 1) ? FN - 1 - idx % FN : idx % FN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[buf][j], xa[buf][i], acc[i][j], 0, 0, 0);
    };
    // slab number i in the order of this tile; those of a last, shorter group in turn
    const bool rotated = turns > 1;
    auto slab_at = [&](int i) { return ((i - kb) | (turns - 1)) < ke - kb ? kb + ((i - kb) ^ turn) : i; };
    // k: the slab that is requested; cur: stage of the one that is multiplied (its fragments are in buffer `buf`), nxt: of the one behind it
    auto slab = [&](auto bufc, int k, int cur, int nxt) {
        constexpr int buf = decltype(bufc)::value;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < READS; ++r) {
            const int lo = r * MFMAS / READS, hi = (r + 1) * MFMAS / READS;
            if (r == BS) {
                wait_loads_and_barrier<(ST - 2) * NL>();   // slab kt + 1 has landed; every wave holds its fragments of slab kt
                __builtin_amdgcn_sched_barrier(0);
            }
            if (r >= BS) {
                const int f0 = 2 * (r - BS);
                for (int f = f0; f < f0 + 2 && f < READS; ++f) read_frag(buf ^ 1, nxt, f);
            }
            mfma_one(buf, lo);
            __builtin_amdgcn_sched_barrier(0);
            if (r >= BS && r - BS < NL) load(cur, r - BS, k);
#pragma unroll
            for (int m = lo + 1; m < hi; ++m) mfma_one(buf, m);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    for (int s = 0; s < ST; ++s) {
        const int k = rotated ? slab_at(kb + s) : kb + s;
#pragma unroll
        for (int j = 0; j < NL; ++j) load(s * SLAB, j, k);
    }
    wait_loads_and_barrier<(ST - 1) * NL>();
#pragma unroll
    for (int r = 0; r < READS; ++r) read_frag(0, 0, r);
    __builtin_amdgcn_sched_barrier(0);
    int cur = 0;
    auto after = [](int s) { return s + SLAB == ST * SLAB ? 0 : s + SLAB; };
    for (int kt = kb; kt < ke; kt += 2) {
        const int n1 = after(cur), n2 = after(n1);
        int k0 = kt + ST, k1 = kt + ST + 1;
        if (rotated) {
            k0 = slab_at(k0);
            k1 = slab_at(k1);
        }
        slab(ic<0>(), k0, cur, n1);
        if (kt + 1 < ke) slab(ic<1>(), k1, n1, n2);
        cur = n2;
    }
    wait_vmem_all();
}

template <int FM, int FN, int ST, bool KTAIL, bool SPLIT>
__global__ __launch_bounds__(kPairThreads) void gemm_nt_pair_kernel(GemmLaunch L) {
    constexpr int BM = 32 * FM, BN = 32 * FN, BK = 64;
    constexpr int R0 = (FM + 1) / 2, R1 = FM - R0;   // fragment rows that group 0 / group 1 finishes
    __shared__ __attribute__((aligned(1024))) char lds[ST * (BM + BN) * BK * 2];
    static_assert(4 * FM * FN * 1024 <= ST * (BM + BN) * BK * 2 && 2 * rect_epilogue_lds(FN) <= ST * (BM + BN) * BK * 2, "exchange and epilogue must fit the ring");
    int t = 0, split = 0, tm, tn;
    if constexpr (SPLIT) {   // the parts of a tile are `tiles` places apart in the sequence
        t = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
        if (t >= L.tiles_m * L.tiles_n * L.splits) return;
        split = t / (L.tiles_m * L.tiles_n);
        t -= split * (L.tiles_m * L.tiles_n);
        tile_at(L, t, tm, tn);
    } else {
        if (FN == 8 && L.p[0].qk_cols > 0 ? !tile_of_block_qk(L, BN, tm, tn) : !tile_of_block(L, tm, tn)) return;
    }
    int turn = 0, turns = 1;
    if (L.take_turns) {
        const int tiles = min(L.tiles_m - tm / L.group_m * L.group_m, L.group_m);
        turns = tiles > 2 ? 4 : tiles;
        turn = (tm % L.group_m + tn) & (turns - 1);
    }
    const GemmParams p = L.p[product_of_tile(L, tm)];
    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w4 = wave & 3;
    const int kb = split * L.slabs_per_split, ke = min((p.K + BK - 1) / BK, kb + L.slabs_per_split);
    f32x4* const ex = reinterpret_cast<f32x4*>(lds) + w4 * (FM * FN * 64) + lane;   // exchange: 64 lanes x 16 bytes per fragment
    auto finish = [&](auto gc, f32x4 (&acc)[FM][FN]) {
        constexpr int G = decltype(gc)::value, OWN0 = G == 0 ? 0 : R0, OWN = G == 0 ? R0 : R1, GIVE0 = G == 0 ? R0 : 0, GIVE = FM - OWN;
        __syncthreads();                       // everyone is done with the ring
#pragma unroll
        for (int i = 0; i < GIVE; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) ex[((GIVE0 + i) * FN + j) * 64] = acc[GIVE0 + i][j];
        __syncthreads();
        f32x4 own[OWN][FN];
#pragma unroll
        for (int i = 0; i < OWN; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) own[i][j] = acc[OWN0 + i][j] + ex[((OWN0 + i) * FN + j) * 64];
        if constexpr (SPLIT) {
            f32x4* dst = reinterpret_cast<f32x4*>(L.partial) + ((static_cast<int64_t>(split) * (L.tiles_m * L.tiles_n) + t) * 4 + w4) * (FM * FN * 64) + lane;
#pragma unroll
            for (int i = 0; i < OWN; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) dst[((OWN0 + i) * FN + j) * 64] = own[i][j];
        } else {
            __syncthreads();                   // the exchange has been read: its LDS is the epilogue's now
            gemm_finish_rect<FM, FN, OWN, FN != 8>(p, own, lds + G * (ST * (BM + BN) * BK), m0, n0, OWN0, w4, lane);
        }
    };
    f32x4 acc[FM][FN];
    if (wave < 4) {
        gemm_pair_slabs<FM, FN, ST, KTAIL, 0>(p, lds, m0, n0, kb, ke, turn, turns, w4, lane, acc);
        finish(ic<0>(), acc);
    } else {
        gemm_pair_slabs<FM, FN, ST, KTAIL, 1>(p, lds, m0, n0, kb, ke, turn, turns, w4, lane, acc);
        finish(ic<1>(), acc);
    }
}

// Second half of a split-K launch: a workgroup per (tile, fragment row) adds the parts in order and runs
// the epilogue on that fragment row of its four waves' sub-tiles.
template <int FM, int FN>
__global__ __launch_bounds__(kGemmThreads) void gemm_reduce_kernel(GemmLaunch L) {
    constexpr int BM = 32 * FM, BN = 32 * FN;
    __shared__ __attribute__((aligned(16))) char lds[rect_epilogue_lds(FN)];
    const int tiles = L.tiles_m * L.tiles_n;
    const int t = blockIdx.x / FM, row = blockIdx.x - t * FM;
    int tm, tn;
    tile_at(L, t, tm, tn);
    const GemmParams p = L.p[product_of_tile(L, tm)];
    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const f32x4* src = reinterpret_cast<const f32x4*>(L.partial) + (static_cast<int64_t>(t) * 4 + wave) * (FM * FN * 64) + row * (FN * 64) + lane;
    const int64_t part = static_cast<int64_t>(tiles) * 4 * (FM * FN * 64);
    f32x4 acc[1][FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[0][j] = src[j * 64];
    for (int s = 1; s < L.splits; ++s) {
        src += part;
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[0][j] += src[j * 64];
    }
    gemm_finish_rect<FM, FN, 1, FN != 8>(p, acc, lds, m0, n0, row, wave, lane);
}

template <int FM, int FN, int ST>
static void launch_pair(const GemmSet& g, int splits, float* partial, hipStream_t st) {
    const int K = g.p[0].K;
    GemmLaunch L = make_launch(g, 32 * FM, 32 * FN);
    L.take_turns = g.n == 1 && weights_from_hbm(g) && (L.tiles_m < 4 || 4 * (g.p[0].M - (L.tiles_m - 1) * 32 * FM) >= 3 * 32 * FM);
    if (splits > 1) {   // (whole slabs only)
        L.slabs_per_split = (K / 64 + splits - 1) / splits;
        L.splits = (K / 64 + L.slabs_per_split - 1) / L.slabs_per_split;
        L.partial = partial;
    }
    if (L.splits > 1) {
        hipLaunchKernelGGL((gemm_nt_pair_kernel<FM, FN, ST, false, true>), dim3(grid_of(L)), dim3(kPairThreads), 0, st, L);
        hipLaunchKernelGGL((gemm_reduce_kernel<FM, FN>), dim3((unsigned)(L.tiles_m * L.tiles_n * FM)), dim3(kGemmThreads), 0, st, L);
    } else if (K % 64 == 0) {
        hipLaunchKernelGGL((gemm_nt_pair_kernel<FM, FN, ST, false, false>), dim3(grid_of(L)), dim3(kPairThreads), 0, st, L);
    } else {
        hipLaunchKernelGGL((gemm_nt_pair_kernel<FM, FN, ST, true, false>), dim3(grid_of(L)), dim3(kPairThreads), 0, st, L);
    }
}

void launch_pair_tiles(int fm, int fn, const GemmSet& g, int splits, float* partial, hipStream_t st) {
#define FLUX_PAIR(FM, FN, ST) if (fm == FM && fn == FN) return launch_pair<FM, FN, ST>(g, splits, partial, st)
    FLUX_PAIR(5, 6, 3); FLUX_PAIR(6, 6, 3); FLUX_PAIR(4, 6, 3); FLUX_PAIR(8, 4, 3); FLUX_PAIR(7, 4, 3); FLUX_PAIR(6, 4, 4);
    FLUX_PAIR(5, 4, 4); FLUX_PAIR(5, 3, 4); FLUX_PAIR(4, 3, 4); FLUX_PAIR(3, 3, 4); FLUX_PAIR(2, 3, 4);
    FLUX_PAIR(2, 2, 6); FLUX_PAIR(4, 8, 3);
#undef FLUX_PAIR
}

}  // namespace flux
