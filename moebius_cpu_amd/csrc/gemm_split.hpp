// EXACT-precision GEMM on the bf16 matrix instructions: every f32 operand is
// split into three bf16 parts (x = hi + mid + lo, each the rounding of what the
// parts before it leave, so the three hold all 24 bits), and a product is the
// sum of the six part products above 2^-24 of it (hi.hi, hi.mid, mid.hi,
// mid.mid, hi.lo, lo.hi), smallest first, summed in f32 by
// v_mfma_f32_16x16x32_bf16. Same operands, conv gathers, prologues and
// epilogues as the f32 kernel of gemm_kernel.hpp.
#pragma once

#include "gemm_kernel.hpp"
#include "split_bf16.hpp"

namespace mh {
namespace gemm {

typedef float floatx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx8s __attribute__((ext_vector_type(8)));

// The split kernel for this GEMM, or false (nothing launched) where the f32
// kernel is to run it (gemm_split_dense.hip, gemm_split_conv.hip).
bool launch_split_dense(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi, int batch);
bool launch_split_dense_pro(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi);
bool launch_split_dense_ln(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi);
bool launch_split_conv(Context &ctx, GemmArgs &p, WeightType wt, int mode, bool pro);

namespace {

constexpr int kSK = 32;  // K per matrix instruction, and per wave group and LDS stage

// One wave's sums on the f32 instructions, straight from memory: rows m.. of A, columns
// n.. and the K values of wave group wk. For tiles with a sum that is infinite or NaN (a
// part product of an infinite value with a zero part is NaN where the f32 product is
// infinite, and a value within half a bf16 step of the largest f32 rounds to an infinite
// part) or too small for its operands' bits (split_bf16.hpp). 2048x1280x1280 of nothing
// but such values: 170 us against 62.
template <int FM, int FN, int WK, int MODE, int PRO, bool F16>
__device__ __forceinline__ void split_redo(const GemmArgs &p, int m, int n, int wk, int lane, floatx4 (&sum)[FM][FN]) {
    const int l16 = lane & 15, kg = lane >> 4;
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(p.a, p.a_bytes);
    const __amdgpu_buffer_rsrc_t a2_rsrc = make_rsrc(p.a2 ? p.a2 : p.a, p.a2 ? p.a2_bytes : p.a_bytes);
    const __amdgpu_buffer_rsrc_t b_rsrc = make_rsrc(p.b, p.b_bytes);
    ConvRow crow[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int row = m + 16 * i + l16;
        if constexpr (MODE >= kConvAligned) crow[i] = conv_row(p, row);
        else crow[i] = ConvRow{PRO == kProAffine ? min(row, p.M - 1) / p.pro_rows : 0, 0, 0, true};
#pragma unroll
        for (int j = 0; j < FN; ++j) sum[i][j] = zero4();
    }
#pragma nounroll
    for (int k0 = wk * kSK; k0 < p.K; k0 += WK * kSK) {
        int tky = 0, tkx = 0, tci = 0;
        if constexpr (MODE == kConvAligned) {
            const int tap = k0 / p.ci;
            tci = k0 - tap * p.ci;
            tky = tap / 3;
            tkx = tap - tky * 3;
        }
        const bool sec = MODE == kDense && p.a2 && k0 >= p.ka;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = k0 + 16 * h + 4 * kg;
            floatx4 a[FM];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                a[i] = sec ? load_a_buf<MODE, PRO>(p, a2_rsrc, crow[i], m + 16 * i + l16, k - p.ka, p.K - p.ka, 0, 0, 0, p.lda2)
                           : load_a_buf<MODE, PRO>(p, a_rsrc, crow[i], m + 16 * i + l16, k, p.K, tky, tkx, tci);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const floatx4 b = load_b_buf<F16>(p, b_rsrc, n + 16 * j + l16, k, p.K);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < FM; ++i) sum[i][j] = Mf<16>::mfma(a[i][t], b[t], sum[i][j]);
            }
        }
    }
}

// WM x WK waves: wave (wm, wk) owns rows [wm * TM, (wm + 1) * TM) of the tile,
// all BN columns and the wk-th 32 of every stage's 32 * WK K values. A rows are
// each read by one wave group only, so they go from memory straight to the
// registers of the lanes that multiply them (16 rows x 128 bytes per load pair)
// and are split there; B goes through LDS already split, one copy for all waves.
// Bound by the splitting and the part products together (the vector and matrix
// pipes both at about 60% in the main loop), and at the UNet's sizes as much by
// what a launch costs around its loop (10 us: first loads, epilogue, drain).
// Against the f32 kernels, in the UNet's step: 8192x1600x320 91 -> 67 us,
// 2048x3200x640 84 -> 70, 512x6400x1280 88 -> 71, 2048x320x2880 55 -> 44, 16 x
// 512x1280x1280 226 -> 142 (190 TFLOP/s; the f32 instructions' rate is 144); the
// step 6.98 -> 6.35 ms. Deeper prefetch, weights split ahead of time (1.5 times the
// bytes to read) and loads straight to LDS measured no faster.
// Two workgroups per CU for WK 1 and 2: one's loads and stores then overlap the
// other's products (2048x3200x640 with WK 2: 69 against 85 us).
template <int TM, int BN, int WM, int WK, int MODE, int PRO, bool F16, int EPI>
__global__ __launch_bounds__(64 * WM * WK, WK <= 2 ? 4 : 2) void gemm_split_kernel(GemmArgs p) {
    constexpr int BM = TM * WM, NT = 64 * WM * WK;
    using L = Waves<BM, BN, WM, 1, WK, 16>;
    constexpr int FM = TM / 16, FN = BN / 16;
    constexpr int SK = kSK * WK;         // K per stage
    constexpr int LS = SK + 8;           // LDS row stride (bf16): rows of a read on distinct banks
    constexpr int NP = F16 ? 2 : 3;      // parts of a B value (an f16 value is two bf16)
    constexpr int PART = BN * LS;        // one part of a stage (bf16)
    constexpr int STAGE = NP * PART;
    constexpr int CPR = SK / 8;          // 8-value chunks per B row
    constexpr int RPP = NT / CPR;        // B rows per load pass
    constexpr int B_LD = (BN + RPP - 1) / RPP;
    const int tiles_m = (p.M + BM - 1) / BM;
    const int tiles_n = (p.N + BN - 1) / BN;
    const TileIdx ti = tile_index(tiles_m, tiles_n);
    if (ti.y) {
        const int64_t bz = ti.y;
        p.a += bz * p.a_bs;
        p.b = static_cast<const char *>(p.b) + bz * p.b_bs * (F16 ? 2 : 4);
        p.out += bz * p.c_bs;
        if (p.res) p.res += bz * p.c_bs;
    }
    constexpr int EPI_F = L::kFixedQuads ? WK * BM * L::CS
                                         : (WK * BM * L::CS > BM * L::CS + 8 * NT ? WK * BM * L::CS : BM * L::CS + 8 * NT);
    constexpr int SMEM = (2 * STAGE / 2 > EPI_F ? 2 * STAGE / 2 : EPI_F);  // floats
    __shared__ __align__(16) float smem[SMEM < 2048 ? 2048 : SMEM];
    __bf16 *const lds = reinterpret_cast<__bf16 *>(smem);

    const SplitSel sel = split_sel();
    const int m0 = ti.tm * BM, n0 = ti.tn * BN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int wm, wn, wk;
    L::index(wave, wm, wn, wk);
    const int l16 = lane & 15, kg = lane >> 4;  // row of a 16-row block, K group of 8
    const int stages = (p.K + SK - 1) / SK;

    // A rows of this lane: byte offset of the row (dense), or its conv geometry
    int aoff[FM], aoff2[FM];
    ConvRow crow[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int row = m0 + wm * TM + i * 16 + l16;
        if constexpr (MODE >= kConvAligned) crow[i] = conv_row(p, row);
        else crow[i] = ConvRow{PRO == kProAffine ? min(row, p.M - 1) / p.pro_rows : 0, 0, 0, true};
        aoff[i] = row < p.M ? int(int64_t(row) * p.lda * 4) : kOob;
        aoff2[i] = row < p.M ? int(int64_t(row) * p.lda2 * 4) : kOob;
    }
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(p.a, p.a_bytes);
    const __amdgpu_buffer_rsrc_t a2_rsrc = make_rsrc(p.a2 ? p.a2 : p.a, p.a2 ? p.a2_bytes : p.a_bytes);
    const __amdgpu_buffer_rsrc_t b_rsrc = make_rsrc(p.b, p.b_bytes);

    // This wave's 32 K values of stage s, eight per lane and row block: lane group
    // kg holds K 4 kg .. 4 kg + 3 and 16 + 4 kg .. 16 + 4 kg + 3 (the same order in
    // B; the sum does not care), so each load of a wave reads 64-byte runs.
    auto fetch_a = [&](int s, floatx4 (&ra)[FM][2]) {
        const int k0 = s * SK + wk * kSK, k = k0 + 4 * kg;
        if constexpr (MODE == kDense) {
            const bool sec = p.a2 && k0 >= p.ka;  // whole groups: ka % 64 == 0
            const int kk = sec ? k - p.ka : k, kend = sec ? p.K - p.ka : p.K;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool in = kk + 16 * h < kend;
                    const int off = in ? (sec ? aoff2[i] : aoff[i]) + (kk + 16 * h) * 4 : kOob;
                    floatx4 v = buf_load4(sec ? a2_rsrc : a_rsrc, off);
                    if constexpr (PRO == kProAffine)
                        v = dense_prologue(p, crow[i].b, k + 16 * h, in && aoff[i] != kOob, v);
                    ra[i][h] = v;
                }
        } else {
            int tky = 0, tkx = 0, tci = 0;
            if constexpr (MODE == kConvAligned) {
                const int tap = k0 / p.ci;
                tci = k0 - tap * p.ci;
                tky = tap / 3;
                tkx = tap - tky * 3;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int kh = k + 16 * h;
                int ky = tky, kx = tkx, c = tci + 4 * kg + 16 * h;
                if constexpr (MODE == kConvVec) {
                    const int tap = kh / p.ci;
                    c = kh - tap * p.ci;
                    ky = tap / 3;
                    kx = tap - ky * 3;
                }
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    const int64_t src = conv_src(p, crow[i], ky, kx);
                    const bool ok = kh < p.K && src >= 0;
                    floatx4 v = buf_load4(a_rsrc, ok ? int((src + c) * 4) : kOob);
                    if constexpr (PRO == kProAffine) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = ok ? prologue1(p, crow[i].b, c + e, v[e]) : 0.0f;
                    }
                    ra[i][h] = v;
                }
            }
        }
    };
    // The same eight K values of B rows brow + RPP i.
    const int brow = tid / CPR, bc = tid % CPR;
    typedef std::conditional_t<F16, halfx8s, floatx8> BV;
    auto fetch_b = [&](int s, BV (&rb)[B_LD]) {
        const int k = s * SK + (bc >> 2) * kSK + 4 * (bc & 3);
#pragma unroll
        for (int i = 0; i < B_LD; ++i) {
            const int n = n0 + brow + RPP * i;
            const bool in = (BN % RPP == 0 || brow + RPP * i < BN) && n < p.N;
            const int64_t e = int64_t(n) * p.ldb + k;
            if constexpr (F16) {
                union {
                    halfx4 q[2];
                    halfx8s v;
                } u;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    u.q[h] = __builtin_bit_cast(
                        halfx4, __builtin_amdgcn_raw_buffer_load_b64(
                                    b_rsrc, in && k + 16 * h < p.K ? int((e + 16 * h) * 2) : kOob, 0, 0));
                rb[i] = u.v;
            } else {
                union {
                    floatx4 q[2];
                    floatx8 v;
                } u;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    u.q[h] = buf_load4(b_rsrc, in && k + 16 * h < p.K ? int((e + 16 * h) * 4) : kOob);
                rb[i] = u.v;
            }
        }
    };
    auto stash_b = [&](int buf, const Split3 (&bs)[B_LD]) {
#pragma unroll
        for (int i = 0; i < B_LD; ++i) {
            if (BN % RPP != 0 && brow + RPP * i >= BN) continue;
            __bf16 *dst = lds + buf * STAGE + (brow + RPP * i) * LS + 8 * bc;
#pragma unroll
            for (int q = 0; q < NP; ++q) *reinterpret_cast<bf16x8 *>(dst + q * PART) = bs[i].q[q].v;
        }
    };

    // hi.hi and, in sums of their own that lose nothing beside the large ones, the
    // five smaller part products
    floatx4 acc[FM][FN], low[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = low[i][j] = zero4();
    const int b_off = l16 * LS + wk * kSK + 8 * kg;
    constexpr int JC = 2;  // column blocks at a time: their products are independent of each other
    constexpr int NC = (FN + JC - 1) / JC;
    auto read_b = [&](int buf, int c, bf16x8 (&b)[JC][NP]) {
        const __bf16 *bs = lds + buf * STAGE + b_off;
#pragma unroll
        for (int j = 0; j < JC; ++j)
            if (c * JC + j < FN)
#pragma unroll
                for (int q = 0; q < NP; ++q)
                    b[j][q] = *reinterpret_cast<const bf16x8 *>(bs + q * PART + (c * JC + j) * 16 * LS);
    };
    // Part products of column blocks c * JC.., smallest first.
    auto products = [&](const Split3 (&a)[FM], int c, const bf16x8 (&b)[JC][NP]) {
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            if (kSplitTerm[t][1] >= NP) continue;
#pragma unroll
            for (int j = 0; j < JC; ++j)
                if (c * JC + j < FN)
#pragma unroll
                    for (int i = 0; i < FM; ++i) {
                        floatx4 &sum = t == 5 ? acc[i][c * JC + j] : low[i][c * JC + j];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].q[kSplitTerm[t][0]].v, b[j][kSplitTerm[t][1]],
                                                                      sum, 0, 0, 0);
                    }
        }
    };
    // Splitting work of a stage in units of one pair: B pairs, then A pairs.
    constexpr int UA = FM * 4, UB = B_LD * 4;
    auto split_units = [&](int lo, int hi, const floatx4 (&ra)[FM][2], Split3 (&a)[FM], const BV (&rb)[B_LD],
                           Split3 (&bs)[B_LD]) {
#pragma unroll
        for (int u = 0; u < UA + UB; ++u) {
            if (u < lo || u >= hi) continue;
            const int i = (u < UB ? u : u - UB) / 4, e = (u < UB ? u : u - UB) % 4;
            if (u < UB)
                split_pair(float(rb[i][2 * e]), float(rb[i][2 * e + 1]), e, sel, bs[i]);
            else
                split_pair(ra[i][e >> 1][2 * (e & 1)], ra[i][e >> 1][2 * (e & 1) + 1], e, sel, a[i]);
        }
    };
    // One stage: the products of the stage in LDS buffer buf with the rows split in
    // a; between them the next stage's values are split (ra -> an, rb -> the other
    // buffer) and the loads after them issued (A two stages ahead, into rf).
    auto stage = [&](int s, int buf, const Split3 (&a)[FM], Split3 (&an)[FM], const floatx4 (&ra)[FM][2],
                     floatx4 (&rf)[FM][2], BV (&rb)[B_LD]) {
        bf16x8 b[2][JC][NP];
        Split3 bs[B_LD];
        read_b(buf, 0, b[0]);
        fetch_a(s + 2, rf);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (c + 1 < NC) read_b(buf, c + 1, b[(c + 1) & 1]);
            products(a, c, b[c & 1]);
            split_units((UA + UB) * c / NC, (UA + UB) * (c + 1) / NC, ra, an, rb, bs);
            constexpr int nm = FM * JC * (NP == 3 ? 6 : 5);
#pragma unroll
            for (int m = 0; m < nm; ++m) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        stash_b(buf ^ 1, bs);
        fetch_b(s + 2, rb);
        __syncthreads();
    };

    // A stage past the end loads zeros; the last stage is multiplied alone.
    floatx4 ra0[FM][2], ra1[FM][2];
    Split3 a0[FM], a1[FM];
    BV rb[B_LD];
    {
        Split3 bs[B_LD];
        fetch_b(0, rb);
        fetch_a(0, ra0);
        fetch_a(1, ra1);
        split_units(0, UB, ra0, a0, rb, bs);
        stash_b(0, bs);
        fetch_b(1, rb);
        split_units(UB, UA + UB, ra0, a0, rb, bs);
        __syncthreads();
    }
    int s = 0;
    for (; s + 2 <= stages; s += 2) {
        stage(s, 0, a0, a1, ra1, ra0, rb);
        stage(s + 1, 1, a1, a0, ra0, ra1, rb);
    }
    if (s < stages) {
        bf16x8 b[2][JC][NP];
        read_b(0, 0, b[0]);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (c + 1 < NC) read_b(0, c + 1, b[(c + 1) & 1]);
            products(a0, c, b[c & 1]);
        }
        __syncthreads();
    }

    __shared__ float ln_st[PRO >= kProLn ? 2 * BM : 1];
    if constexpr (PRO == kProLnPart) ln_stats_from_parts<BM, NT>(p, m0, ln_st);
    SplitProbe probe;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 4; v += 2) {
                acc[i][j][v] = acc[i][j][v] + low[i][j][v];
                acc[i][j][v + 1] = acc[i][j][v + 1] + low[i][j][v + 1];
                probe.see(acc[i][j][v], acc[i][j][v + 1]);
            }
    auto redo = [&](floatx4 (&sum)[FM][FN]) {
        // the lane's number again, so that nothing this derives from it is kept through the loop
        int lane2 = lane;
        asm volatile("" : "+v"(lane2));
        split_redo<FM, FN, WK, MODE, PRO, F16>(p, m0 + wm * TM, n0, wk, lane2, sum);
    };
    write_tile<BM, BN, WM, 1, WK, 16, EPI, false>(p, smem, acc, m0, n0, 0, PRO >= kProLn ? ln_st : nullptr,
                                                  probe.bad(), redo);
}

// The tilings: rows per wave, columns, waves over the rows, wave groups over K;
// and a tiling's time as measured over the UNet's and VAE's GEMMs inside their
// passes (60 shapes, M 256..8192, N 320..6400, K 320..5760): `launch` us for a
// launch, its first loads and its epilogue, then per round of one workgroup per CU
// `round` us and `per_k` ns for each element of K (7% rms). The wave groups over K
// shorten a round by as much as they shorten its tile, so they serve the grids of
// about one round; 128x80 runs the products at 200 TFLOP/s, 32x48 at 130.
struct SplitTile {
    int tm, bn, wm, wk;
    float launch, round, per_k;
};
constexpr SplitTile kSplitTiles[] = {
    {16, 80, 8, 1, 10.7f, 1.9f, 26.3f}, {16, 64, 8, 1, 10.3f, 1.4f, 22.1f}, {16, 80, 4, 2, 14.0f, 0.3f, 17.8f},
    {16, 64, 4, 2, 10.1f, 0.5f, 14.4f}, {16, 48, 4, 2, 10.0f, 1.0f, 10.5f}, {16, 80, 2, 4, 6.4f, 4.6f, 10.4f},
    {16, 64, 2, 4, 7.4f, 3.4f, 9.0f},   {16, 48, 2, 4, 9.0f, 1.6f, 5.9f},   {16, 32, 2, 4, 11.7f, 1.2f, 4.4f},
};
constexpr int kSplitCount = int(sizeof(kSplitTiles) / sizeof(kSplitTiles[0]));

struct SplitPlan {
    int tm = 0, bn = 0, wm = 0, wk = 0;
};

// The tiling of the least modelled time, or tm = 0 for the f32 kernel where that
// is no more than the f32 kernels' (11.5 us and 116 TFLOP/s fit the same shapes within
// 10%). The sum over the UNet's GEMMs comes within 0.5% of the best choice for each.
// Loops shorter than the shapes' (K under 256) need 3% less: 8820x556x96 18.5 against
// 16.6 us in f32, 994x2665x176 16.6 against 16.1; of 1044 random shapes that take the
// split kernel two are 3 to 4% slower in it, and all 1.5 times faster on average.
// Kept by the f32 kernels: under 0.8 GFLOP, where fixed costs decide (4096x256x128
// 7.5 against 6.5 us, 64x1280x1280 11.1 against 10.4), and small grids of long K,
// which they split over workgroups (256x640x5760 44 against 35 us). Up to 32 rows of a
// large weight (the time projections) are bound by reading it: the narrowest tile
// whose columns are one round of the CUs, over weights not yet in the caches: 2x8192x1024
// 11.9 us (32 columns) against 13.4, 2x11200x1280 15.2 (48) against 17.8, 32x16384x1280
// 20.9 (64) against 23.5, 2x20480x1280 21.6 (80) against 26.5, 16x1280x11520 64 against
// 84; not past that round (2x25600x1280 34 against 31) or under K = 768 (32x16384x512
// 11.6 against 11.2), and not the convs, whose K the f32 kernels split over workgroups
// (an 8x8 map's stride 2, 16x1280x11520: 78 against 54 us). Convs leave 64x80 with two wave groups out: the
// gather's addresses spill there (64x64 x 320 channels 86 us, 64x48 69, f32 80).
// gn_rows: the rows per item where the output's GroupNorm partials are wanted (0: not);
// a tile height that does not divide them costs the next GroupNorm a statistics launch
// (priced, 1568x512x512 and the GroupNorm's fold take 17.5 us for 19.6, 2592 rows 23.0 for
// 24.3, 3136 26.7 for 26.6).
inline SplitPlan plan_split(int64_t M, int64_t N, int64_t K, int cus, int batch, bool conv, int gn_rows) {
    if (M <= 32 && K >= 768 && N * K >= (int64_t(1) << 23) && batch == 1 && !conv)
        for (const int bn : {32, 48, 64, 80})
            if (ceil_div(N, int64_t(bn)) <= cus) return SplitPlan{16, bn, 2, 4};
    const double products = double(M) * double(N) * double(K) * batch;
    if (products < 4e8) return SplitPlan{};
    // the statistics launch of a tiling whose rows would straddle items
    auto stats = [&](int64_t rows) { return gn_rows && gn_rows % rows ? 5.0 + double(M * N) * 4.0 / 4.5e6 : 0.0; };
    SplitPlan best;
    double cost = (11.5 + products * (2.0 / 116e6)) * (K < 256 ? 0.97 : 1.0) + stats(32);
    for (const SplitTile &t : kSplitTiles) {
        if (conv && t.bn == 80 && t.wk == 2) continue;
        const int64_t tiles = ceil_div(M, int64_t(t.tm) * t.wm) * ceil_div(N, int64_t(t.bn)) * batch;
        const double c = t.launch + double(ceil_div(tiles, int64_t(cus))) * (t.round + t.per_k * 1e-3 * double(K)) +
                         stats(t.tm * t.wm);
        if (c < cost) best = SplitPlan{t.tm, t.bn, t.wm, t.wk}, cost = c;
    }
    return best;
}

// The same under the context's tuning (gemm_split; gemm_plan forces an f32 tiling).
inline SplitPlan split_plan_for(const Context &ctx, int64_t M, int N, int K, int batch, bool conv, int gn_rows = 0) {
    ShapePlan forced;
    if (!ctx.tune.gemm_split || K % 4 || forced_plan(ctx.tune, int(M), N, K, forced)) return SplitPlan{};
    if (ctx.tune.split_tm) return SplitPlan{ctx.tune.split_tm, ctx.tune.split_bn, ctx.tune.split_wm, ctx.tune.split_wk};
    return plan_split(M, N, K, ctx.cu_count, batch, conv, gn_rows);
}

template <int TM, int BN, int WM, int WK, int MODE, int PRO, bool F16>
void launch_split_cfg(Context &ctx, GemmArgs &p, GemmEpilogue epi, int batch) {
    constexpr int BM = TM * WM, NT = 64 * WM * WK;
    static_assert(BM >= 32 && BN >= 32, "the callers' buffers hold a GroupNorm partial per 32 rows and a LayerNorm "
                                        "partial per 32 columns");
    constexpr bool kSquare = Waves<BM, BN, WM, 1, WK, 16>::kFixedQuads;
    const unsigned tiles = unsigned(ceil_div(p.M, BM) * ceil_div(p.N, BN));
    log_gemm(ctx, "split", p, BM, BN, 1, MODE, PRO, F16, epi, batch, WM, 1, WK);
    const GemmTimer timer(ctx, "f32 split", p, BM, BN, WM, 1, WK, 1, MODE, batch);
    p.k_split = p.K;
    p.vec_out = out_vec_ok(p, BM);
    gn_partials_plan(p, BM, BN, 1, batch, kSquare);
    ln_partials_plan(p, BN, 1, batch);
    const dim3 grid(tiles, unsigned(batch));
    if constexpr (MODE == kDense) {
        if (epi == GemmEpilogue::Silu) {
            gemm_split_kernel<TM, BN, WM, WK, MODE, PRO, F16, 1><<<grid, NT, 0, ctx.stream>>>(p);
            MH_LAUNCH_CHECK();
            return;
        }
    } else {
        MH_REQUIRE(epi == GemmEpilogue::None, "conv GEMM: SiLU epilogue not available");
    }
    gemm_split_kernel<TM, BN, WM, WK, MODE, PRO, F16, 0><<<grid, NT, 0, ctx.stream>>>(p);
    MH_LAUNCH_CHECK();
}

template <int I, int MODE, int PRO, bool F16>
bool launch_split_tile(Context &ctx, GemmArgs &p, const SplitPlan &s, GemmEpilogue epi, int batch) {
    if constexpr (I < kSplitCount) {
        constexpr SplitTile t = kSplitTiles[I];
        if (s.tm == t.tm && s.bn == t.bn && s.wm == t.wm && s.wk == t.wk) {
            launch_split_cfg<t.tm, t.bn, t.wm, t.wk, MODE, PRO, F16>(
                ctx, p, epi, batch);
            return true;
        }
        return launch_split_tile<I + 1, MODE, PRO, F16>(ctx, p, s, epi, batch);
    }
    return false;
}

// A vector A operand (checked by the caller) and vector weight rows.
template <int MODE, int PRO>
bool launch_split(Context &ctx, GemmArgs &p, WeightType wt, GemmEpilogue epi, int batch) {
    const SplitPlan s = split_plan_for(ctx, p.M, p.N, p.K, batch, MODE >= kConvAligned, p.gnp ? p.gn_item_rows : 0);
    const int esz = wt == kF16 ? 2 : 4;
    if (!s.tm || p.ldb % 4 || reinterpret_cast<uintptr_t>(p.b) % (4 * esz) || (batch > 1 && p.b_bs % 4)) return false;
    return wt == kF16 ? launch_split_tile<0, MODE, PRO, true>(ctx, p, s, epi, batch)
                      : launch_split_tile<0, MODE, PRO, false>(ctx, p, s, epi, batch);
}

}  // namespace
}  // namespace gemm
}  // namespace mh
