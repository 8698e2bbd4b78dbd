// Winograd F(2x2, 3x3) conv in one kernel (src/engine/winograd.rs:48-120):
// the input transform, the 16 plane products and the output transform of a
// block of 64 tiles x 64 output channels stay on chip, so V and M (16 planes
// of tiles x channels each) never reach HBM. The separate path writes and
// reads both: about 4.2 GB per 512x512x128 conv of the VAE decoder.
//
// Workgroup: 512 threads, one per CU (LDS: two V stages of 64 KB), walking a
// share of the (channel block, tile block) items. Per chunk of 16 input channels
// every thread transforms one tile's 4x4 patch for two channels (the reference's
// operation order, as wino_input_kernel) into the V stage [plane][tile][channel];
// the 8 channel pairs of a tile sit on adjacent lanes, so a patch load reads
// 64-byte runs. Wave w (of 8, two per SIMD) multiplies planes 2w and 2w + 1 on
// v_mfma_f32_32x32x16_bf16 with both operands split in three bf16 parts
// (split_bf16.hpp): V from LDS in f32, split by the one wave that reads it, U from
// global memory (L2 resident) split at load and packed so that every load of a wave
// is one run of 1 KB. At the end the planes go through LDS, half the tiles at a
// time, and each thread applies the output transform (winograd.rs:329-352, as
// wino_output_kernel) to one tile and four channels, adding bias and the optional
// residual.
//
// What bounds it (MI355X, 512x512x128 -> 128, parts taken out of a copy, all on one
// board): the products alone 130 us, with the transforms 148, with the patch and U
// loads 221, with the output transform and its stores 279 (257 for a whole call on
// others); on the f32 instructions the same conv took 358 us, its products alone 239. The loads cost what they do because
// the vector L1 serves 96 KB of U and 64 KB of patches per chunk and workgroup:
// 64 tiles per workgroup, twice what the f32 kernel took, halve U's share, and
// 128 accumulators per lane are what that leaves room for. The registers are full:
// a few more live values spill the patch in the loop (392 us), so the output
// transform's numbers are derived anew from the thread's, the patch's validity is
// kept in scalar masks and the next item's loads wait for the sums to leave.
// 128x128x512 -> 512: 402 us in f32, 230 to 251 here. VAE decode 12.97 -> 9.77 ms.
#include <algorithm>

#include "common.hpp"
#include "dmath.hpp"
#include "kernels.hpp"
#include "split_bf16.hpp"

namespace mh {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr int kFT = 64;        // tiles per workgroup
constexpr int kFC = 64;        // output channels per workgroup
constexpr int kFK = 16;        // input channels per chunk: one matrix instruction's K
constexpr int kVStage = 16 * kFT * kFK;  // floats; 16-byte quads of a row swizzled (vquad)
constexpr int kHT = kFT / 2;             // tiles per half of the M exchange
constexpr int kMS = kFC + 4;             // M row stride in LDS (floats)
constexpr int kRed = 16 * kHT * kMS;     // GroupNorm reduction scratch, past the M exchange
constexpr int kLds = kRed + 2 * 8 * 64;  // floats, 140 KB
static_assert(2 * kVStage <= kLds && kRed >= kVStage, "the V stages fit, the scratch in stage 1 or past it");
constexpr uint32_t kXEnd = 0x80000000u;  // the input buffer's extent
constexpr int kOob = int(kXEnd);         // past any buffer: reads zero
constexpr int kUBlk = 1024;              // bytes of one packed U block: 32 channels x 16 K of one part

struct FGeo {
    int h, w, hi, wi, th, tw;
    int tiles;  // the input's 2 GiB hold no more than 2^24 pixels
};

struct FArgs {
    const float *x;
    const char *u;  // packed (wino_u_fused_kernel)
    const float *psc, *psh, *bias, *res2;
    float *out, *gnp;
    int *sick;       // per workgroup: whether it met a sum to be redone (SplitProbe)
    const float *w;  // [16][co][ci], the U that u holds split
    FGeo g;
    uint32_t u_bytes;
    int ci, co, psilu, nco_blocks, nwork;
    int gn_halves;  // partials of 32 tiles each, not of a whole block: items of an odd number of 32 tiles
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), short(0), int(bytes), 0x00020000);
}

__device__ __forceinline__ floatx4 sub4(floatx4 a, floatx4 b) { return floatx4{a[0] - b[0], a[1] - b[1], a[2] - b[2], a[3] - b[3]}; }
__device__ __forceinline__ floatx4 add4(floatx4 a, floatx4 b) { return floatx4{a[0] + b[0], a[1] + b[1], a[2] + b[2], a[3] + b[3]}; }

constexpr int kFThreads = 512;  // 8 waves, two per SIMD
constexpr int kFPlanes = 16 / (kFThreads / 64);  // planes per wave

// Where quad q (4 channels) of tile row t sits in its 64-byte V row: rows four
// apart take different banks.
__device__ __forceinline__ int vquad(int t, int q) { return (q ^ ((t >> 2) & 3)) * 4; }

// F32: the repair, launched after each conv and done at once where no workgroup
// flagged its sums. A part product of an infinite value with a zero part is NaN where
// the f32 product is infinite, and a value within half a bf16 step of the largest f32
// rounds to an infinite part; and the sums of operands below 2^-110 lack bits
// (split_bf16.hpp). So a workgroup that met such a sum does its items again, products,
// outputs and GroupNorm partials, on v_mfma_f32_32x32x2f32 with the unsplit operands
// (256x256x128 -> 128, every value NaN: 195 us for both, 94 for the conv alone; the
// residual is read again, so it is not the output).
template <int UP, bool PRO, bool F32>
__global__ __launch_bounds__(kFThreads, 2) void wino_fused_kernel(FArgs a) {
    if constexpr (F32)
        if (!a.sick[blockIdx.x]) return;
    const FGeo &g = a.g;
    const int ci = a.ci, co = a.co, nwork = a.nwork;
    __shared__ __align__(16) float lds[kLds];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const SplitSel sel = split_sel();
    // Work items (channel block, tile block), channel block outer. Workgroup i
    // runs on XCD i % 8 (round-robin dispatch); each XCD takes one contiguous
    // eighth of the items, so it works through few channel blocks and their U
    // panels stay in its L2, and its workgroups take every (grid / 8)-th item
    // of that range. The grid holds one workgroup per CU, and a workgroup
    // issues its next item's first patch and U loads once the current item's
    // sums have left their registers, half way through its output transform.
    const int ntb = nwork / a.nco_blocks;
    const int per_xcd = (nwork + 7) / 8;
    const int slots = int(gridDim.x) / 8;
    const int item_end = min(nwork, (int(blockIdx.x) % 8 + 1) * per_xcd);
    const int first = (int(blockIdx.x) % 8) * per_xcd + int(blockIdx.x) / 8;
    if (first >= item_end) {
        if (!F32 && tid == 0) a.sick[blockIdx.x] = 0;
        return;
    }
    const __amdgpu_buffer_rsrc_t ur = rsrc(a.u, a.u_bytes);
    const int per_item = g.th * g.tw;
    const int n_items = g.tiles / per_item;

    // Producer role (every thread): tile vt of the block, channel pair vq of the
    // chunk; the 8 pairs of a tile sit on 8 adjacent lanes (64-byte runs).
    const int vq = tid & (kFK / 2 - 1), vt = tid >> 3;
    // Consumer role: wave w, planes kFPlanes w .. + kFPlanes - 1, two 32-tile by two
    // 32-channel blocks. Lane l holds row l % 32, K 8 (l / 32) .. + 7 of the chunk.
    const int row = lane & 31, kg = lane >> 5;
    // Per item: the block's first tile and channel; the producer's source pixel, which
    // of its patch's rows and columns (at -1, 0, 1, 2 from it, at -1, 0, 0, 1 when
    // upsampling) are inside the image, and its batch item; the wave's first U block
    // (kUBlk bytes each, plane-major [plane][ci / 16][co / 32][part]).
    int t0 = 0, co0 = 0, vb = 0, ubase = 0;
    int porg = 0;                   // bytes of source pixel (sy, sx), channel 2 vq; the buffer starts a row and a
    bool rowin[4], colin[4];        // pixel early, so that a patch row or column's step is never negative
    const int prow = g.w * ci * 4, pcol = ci * 4;  // bytes per source row, per pixel
    constexpr int kStep[4] = {0, 1, 2 - UP, 3 - UP};  // patch row / column k -> source offset + 1
    // A load's checked offset is porg or kOob; the patch's step and the chunk are in its
    // scalar offset. With the extent at kXEnd whatever the map, kOob is out of range
    // whether the check leaves the scalar offset out, adds it or takes it off the extent
    // (which on a map of a row or two it exceeds), and the loads that are made are inside
    // the input by rowin and colin alone.
    const __amdgpu_buffer_rsrc_t xr = rsrc(reinterpret_cast<const char *>(a.x) - prow - pcol, kXEnd);
    auto setup_producer = [&](int it) {
        int ptid = tid;
        asm volatile("" : "+v"(ptid));
        const int tv = it % ntb * kFT + (ptid >> 3);
        const int b = tv / per_item, rem = tv - b * per_item;
        const int ty = rem / g.tw, tx = rem - ty * g.tw;
        vb = min(b, n_items - 1);  // a tile past the end reads nothing, but keeps its prologue loads in range
        const int sy = (2 * ty) >> UP, sx = (2 * tx) >> UP;
        porg = int(uint32_t((b * g.h + sy) * g.w + sx) * uint32_t(pcol)) + 8 * (ptid & (kFK / 2 - 1));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int iy = 2 * ty + k - 1, ix = 2 * tx + k - 1;
            rowin[k] = tv < g.tiles && iy >= 0 && iy < g.hi;
            colin[k] = ix >= 0 && ix < g.wi;
        }
    };
    auto setup_consumer = [&](int it) {
        t0 = it % ntb * kFT;
        co0 = (it / ntb) * kFC;
        ubase = ((kFPlanes * wave * (ci / kFK)) * (co / 32) + co0 / 32) * 3 * kUBlk;
    };
    floatx2 d[16];
    auto produce = [&](int kc) {
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
            d[kk] = __builtin_bit_cast(
                floatx2, __builtin_amdgcn_raw_buffer_load_b64(
                             xr, rowin[kk >> 2] && colin[kk & 3] ? porg : kOob,
                             kStep[kk >> 2] * prow + kStep[kk & 3] * pcol + kc * kFK * 4, 0));
    };
    auto transform_store = [&](int kc, int stage) {
        if constexpr (PRO) {
            const int c = kc * kFK + 2 * vq;
            const floatx2 sc = *reinterpret_cast<const floatx2 *>(a.psc + int64_t(vb) * ci + c);
            const floatx2 sh = *reinterpret_cast<const floatx2 *>(a.psh + int64_t(vb) * ci + c);
#pragma unroll
            for (int kk = 0; kk < 16; ++kk) {
                if (rowin[kk >> 2] && colin[kk & 3]) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float y = __builtin_fmaf(d[kk][e], sc[e], sh[e]);
                        if (a.psilu) y = ref_silu(y);
                        d[kk][e] = y;
                    }
                }
            }
        }
        floatx2 tt[16];
#pragma unroll
        for (int col = 0; col < 4; ++col) {
            const floatx2 d0 = d[col], d1 = d[4 + col], d2 = d[8 + col], d3 = d[12 + col];
            tt[col] = d0 - d2;
            tt[4 + col] = d1 + d2;
            tt[8 + col] = d2 - d1;
            tt[12 + col] = d1 - d3;
        }
        float *vs = lds + stage * kVStage + vt * kFK + vquad(vt, vq >> 1) + 2 * (vq & 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const floatx2 *q = tt + r * 4;
            *reinterpret_cast<floatx2 *>(vs + (r * 4) * kFT * kFK) = q[0] - q[2];
            *reinterpret_cast<floatx2 *>(vs + (r * 4 + 1) * kFT * kFK) = q[1] + q[2];
            *reinterpret_cast<floatx2 *>(vs + (r * 4 + 2) * kFT * kFK) = q[2] - q[1];
            *reinterpret_cast<floatx2 *>(vs + (r * 4 + 3) * kFT * kFK) = q[1] - q[3];
        }
    };

    floatx16 acc[kFPlanes][2][2];  // [plane][tile block][channel block]
    static_assert(kFPlanes == 2, "two planes per wave, taken in turn");
    // U parts of plane p, chunk kc: six whole blocks.
    auto load_u = [&](int p, int kc, bf16x8 (&dst)[2][3]) {
        const int off = ubase + ((p * (ci / kFK) + kc) * (co / 32)) * 3 * kUBlk;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 3; ++q)
                dst[j][q] = __builtin_bit_cast(
                    bf16x8, __builtin_amdgcn_raw_buffer_load_b128(ur, lane * 16, off + (j * 3 + q) * kUBlk, 0));
    };
    const int vlo = (kFPlanes * wave * kFT + row) * kFK + vquad(row, 2 * kg);
    const int vhi = (kFPlanes * wave * kFT + row) * kFK + vquad(row, 2 * kg + 1);
    // V rows of plane p, tile block i from LDS, split.
    auto read_v = [&](const float *vs, int p, int i, Split3 &v) {
        // rows 32 apart share their swizzle
        const floatx4 lo = *reinterpret_cast<const floatx4 *>(vs + vlo + (p * kFT + 32 * i) * kFK);
        const floatx4 hi = *reinterpret_cast<const floatx4 *>(vs + vhi + (p * kFT + 32 * i) * kFK);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            split_pair(e < 2 ? lo[2 * e] : hi[2 * e - 4], e < 2 ? lo[2 * e + 1] : hi[2 * e - 3], e, sel, v);
    };
    auto products = [&](int p, int i, const Split3 &v, const bf16x8 (&uu)[2][3]) {
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[p][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v.q[kSplitTerm[t][0]].v,
                                                                      uu[j][kSplitTerm[t][1]], acc[p][i][j], 0, 0, 0);
    };
    // The same on the f32 instructions: lane l holds K 4 (l / 32) .. + 3 of each half
    // chunk, one of them per instruction.
    auto products_f32 = [&](const float *vs, int kc) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int p = 0; p < kFPlanes; ++p) {
                floatx4 va[2], ub[2];
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    va[i] = *reinterpret_cast<const floatx4 *>(vs + ((kFPlanes * wave + p) * kFT + 32 * i + row) * kFK +
                                                               vquad(row, 2 * s + kg));
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    ub[j] = *reinterpret_cast<const floatx4 *>(
                        a.w + (int64_t(kFPlanes * wave + p) * co + co0 + 32 * j + row) * ci + kc * kFK + 8 * s + 4 * kg);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[p][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[i][t], ub[j][t], acc[p][i][j], 0, 0, 0);
            }
    };
    const int nk = ci / kFK;
    bool sick = false;
    int item = first;
    setup_producer(item);
    setup_consumer(item);
    bf16x8 u0[2][3], u1[2][3];
    produce(0);
    if constexpr (!F32) load_u(0, 0, u0);
    for (;;) {
        const int next = item + slots;
        const bool has_next = next < item_end;
        transform_store(0, 0);
        produce(1);
#pragma unroll
        for (int p = 0; p < kFPlanes; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[p][i][j][v] = 0.f;
        __syncthreads();
        // Four steps of twelve products per chunk, each with the split of the next
        // step's V between them, the last with the next chunk's transform. The loads
        // are spread over the chunk and waited for in issue order: the patch of the
        // chunk after next once the transform has used its registers, the second
        // plane's U at the start of the chunk, the next chunk's first U half way.
        for (int kc = 0; kc < nk; ++kc) {
            const float *vs = lds + (kc & 1) * kVStage;
            if constexpr (F32) {
                products_f32(vs, kc);
            } else {
                load_u(1, kc, u1);
                __builtin_amdgcn_sched_barrier(0);
                Split3 v;
                read_v(vs, 0, 0, v);
                products(0, 0, v, u0);
                __builtin_amdgcn_sched_barrier(0);
                read_v(vs, 0, 1, v);
                products(0, 1, v, u0);
                __builtin_amdgcn_sched_barrier(0);
                load_u(0, min(kc + 1, nk - 1), u0);
                read_v(vs, 1, 0, v);
                products(1, 0, v, u1);
                __builtin_amdgcn_sched_barrier(0);
                read_v(vs, 1, 1, v);
                products(1, 1, v, u1);
            }
            if (kc + 1 < nk) transform_store(kc + 1, (kc + 1) & 1);
            if (kc + 2 < nk) produce(kc + 2);
            __syncthreads();
        }
        const int et0 = t0, eco0 = co0;
        // the thread's number again, so that nothing the output transform derives from
        // it is kept in registers through the products
        int etid = tid;
        asm volatile("" : "+v"(etid));
        const int elane = etid & 63;
        float *const mw = lds + (kFPlanes * wave * kHT + 4 * (elane >> 5)) * kMS + (elane & 31);
        floatx4 gs{0.f, 0.f, 0.f, 0.f}, gq = gs;  // GroupNorm sums of the values stored
        // GroupNorm partials of this block or of each half (per channel: sum and sum of
        // squares over its 256 or 128 pixels), for the next GroupNorm's fold in place of
        // a statistics pass: the four threads of a wave that hold channel quad q (tiles
        // 4w .. 4w + 3 of each half) by xor butterfly, then the eight waves in order
        // through LDS past the M exchange.
        auto write_partials = [&](int block) {
#pragma unroll
            for (int off = 16; off < 64; off <<= 1)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    gs[e] += __shfl_xor(gs[e], off, 64);
                    gq[e] += __shfl_xor(gq[e], off, 64);
                }
            floatx4 *red = reinterpret_cast<floatx4 *>(lds + kRed);
            if (elane < kFC / 4) {
                red[wave * (kFC / 4) + elane] = gs;
                red[(kFThreads / 64 + wave) * (kFC / 4) + elane] = gq;
            }
            __syncthreads();
            if (etid < kFC / 4) {
                floatx4 ts = red[etid], tq = red[(kFThreads / 64) * (kFC / 4) + etid];
#pragma unroll
                for (int w8 = 1; w8 < kFThreads / 64; ++w8) {
                    ts = add4(ts, red[w8 * (kFC / 4) + etid]);
                    tq = add4(tq, red[(kFThreads / 64 + w8) * (kFC / 4) + etid]);
                }
                float *dst = a.gnp + (int64_t(block) * co + eco0 + 4 * etid) * 2;
                *reinterpret_cast<floatx4 *>(dst) = floatx4{ts[0], tq[0], ts[1], tq[1]};
                *reinterpret_cast<floatx4 *>(dst + 4) = floatx4{ts[2], tq[2], ts[3], tq[3]};
            }
        };
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            // M [16][tile][channel] of 32 tiles through LDS: register v of lane l holds
            // row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32 of its block.
            if (half) __syncthreads();  // the first half's reads are done
#pragma unroll
            for (int p = 0; p < kFPlanes; ++p)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        mw[(p * kHT + 8 * (v >> 2) + (v & 3)) * kMS + 32 * j] = acc[p][half][j][v];
            if (half) {  // the sums have left their registers: the next item's first loads (the last item's
                         // again at the end, so that nothing older stays live)
                setup_consumer(has_next ? next : item);
                setup_producer(has_next ? next : item);
                if constexpr (!F32) load_u(0, 0, u0);
                produce(0);
            }
            __syncthreads();
            const int tl = etid >> 4, q = etid & 15;
            const int t = et0 + kHT * half + tl;
            if (t < g.tiles) {
                const int b = t / per_item, rem = t - b * per_item;
                const int ty = rem / g.tw, tx = rem - ty * g.tw;
                const float *src = lds + tl * kMS + 4 * q;
                floatx4 m0[4], m1[4];
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) {
                    const floatx4 aa = *reinterpret_cast<const floatx4 *>(src + (rr * 4) * kHT * kMS);
                    const floatx4 bb = *reinterpret_cast<const floatx4 *>(src + (rr * 4 + 1) * kHT * kMS);
                    const floatx4 cc = *reinterpret_cast<const floatx4 *>(src + (rr * 4 + 2) * kHT * kMS);
                    const floatx4 dd = *reinterpret_cast<const floatx4 *>(src + (rr * 4 + 3) * kHT * kMS);
                    m0[rr] = add4(add4(aa, bb), cc);
                    m1[rr] = sub4(sub4(bb, cc), dd);
                    asm volatile("" ::: "memory");  // sixteen rows at once would not fit the registers
                }
                const int c = eco0 + 4 * q;
                const floatx4 bv = a.bias ? *reinterpret_cast<const floatx4 *>(a.bias + c) : floatx4{0.f, 0.f, 0.f, 0.f};
                floatx4 y[4];
                y[0] = add4(add4(m0[0], m0[1]), m0[2]);
                y[1] = add4(add4(m1[0], m1[1]), m1[2]);
                y[2] = sub4(sub4(m0[1], m0[2]), m0[3]);
                y[3] = sub4(sub4(m1[1], m1[2]), m1[3]);
                if constexpr (!F32) {
                    // The largest of the tile's four pixels in each channel: every plane is in
                    // one of them, and a small one beside it is a difference of its terms.
                    float top[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        top[e] = abs_max(abs_max(y[0][e], y[1][e]), abs_max(y[2][e], y[3][e]));
                    SplitProbe probe;
                    probe.see(top[0], top[1]);
                    probe.see(top[2], top[3]);
                    sick = sick || probe.bad();
                }
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) y[kk] = add4(y[kk], bv);
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    const int oy = 2 * ty + (kk >> 1), ox = 2 * tx + (kk & 1);
                    if (oy >= g.hi || ox >= g.wi) continue;
                    const int64_t o = int64_t((b * g.hi + oy) * g.wi + ox) * co + c;
                    floatx4 rv = y[kk];
                    if (a.res2) rv = add4(rv, *reinterpret_cast<const floatx4 *>(a.res2 + o));
                    *reinterpret_cast<floatx4 *>(a.out + o) = rv;
                    if (a.gnp) {
                        gs = add4(gs, rv);
#pragma unroll
                        for (int e = 0; e < 4; ++e) gq[e] = __builtin_fmaf(rv[e], rv[e], gq[e]);
                    }
                }
            }
            if (a.gnp && a.gn_halves && et0 + kHT * half < g.tiles) {
                write_partials(et0 / kHT + half);
                gs = gq = floatx4{0.f, 0.f, 0.f, 0.f};
            }
        }
        if (a.gnp && !a.gn_halves) write_partials(et0 / kFT);
        if (!has_next) break;
        __syncthreads();  // the output transform's reads of M are done before V stage 0 is written
        item = next;
    }
    if constexpr (!F32) {
        const int bad = __syncthreads_or(sick);
        if (tid == 0) a.sick[blockIdx.x] = bad;
    }
}

// u [16][co][ci] -> packed [16][ci / 16][co / 32][part][lane][8]: lane l of a block
// holds channel l % 32, K 8 (l / 32) .. + 7. An infinite value, or one that rounds to
// infinity, makes the sums of its channel infinite or NaN, and the repair reads u.
__global__ void wino_u_fused_kernel(const float *__restrict__ u, int co, int ci, char *__restrict__ uf) {
    const SplitSel sel = split_sel();
    const int64_t blocks = int64_t(16) * (ci / kFK) * (co / 32);
    for (int64_t e = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; e < blocks * 64;
         e += int64_t(gridDim.x) * blockDim.x) {
        const int lane = int(e & 63);
        const int64_t blk = e >> 6;
        const int cb = int(blk % (co / 32));
        const int64_t r = blk / (co / 32);
        const int kc = int(r % (ci / kFK)), plane = int(r / (ci / kFK));
        const float *src = u + (int64_t(plane) * co + cb * 32 + (lane & 31)) * ci + kc * kFK + 8 * (lane >> 5);
        Split3 s;
#pragma unroll
        for (int p = 0; p < 4; ++p) split_pair(src[2 * p], src[2 * p + 1], p, sel, s);
        char *dst = uf + blk * 3 * kUBlk + lane * 16;
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8 *>(dst + q * kUBlk) = s.q[q].v;
    }
}

template <int UP, bool PRO>
void launch_fused(Context &ctx, const FArgs &a) {
    // one workgroup per CU (its LDS holds one), a multiple of 8 (see the work
    // order in the kernel), no more than the items of one XCD's share need
    const int64_t per_xcd = ceil_div(a.nwork, 8);
    const unsigned grid = unsigned(8 * std::max<int64_t>(1, std::min<int64_t>(ctx.cu_count / 8, per_xcd)));
    wino_fused_kernel<UP, PRO, false><<<grid, kFThreads, 0, ctx.stream>>>(a);
    MH_LAUNCH_CHECK();
    wino_fused_kernel<UP, PRO, true><<<grid, kFThreads, 0, ctx.stream>>>(a);
}

// Where this kernel is faster than the three (whose plane GEMM runs at about 150
// TFLOP/s in split products), both modelled in us. This one: rounds of one workgroup
// per CU, 3.6 us for each 16 input channels and 6 for the output transform, 8 for
// the two launches, and the weights' reordering where the caller has no copy. The
// three: V and M of 16 planes at 4 TB/s, the products, 12 for the launches. A round
// that is nearly empty costs as much as a full one, so the line is no tile count.
// Whole calls, the weights reordered in them, three kernels -> one: 2x64x64x512, one
// round, 137 -> 124 us; 64x64x512, half a round, 76 -> 115; 108x148x256 89 -> 66;
// 512x512x128, 8 rounds, 580 -> 257; 128x128x512, 2 rounds, 276 -> 230; 130x130x512,
// one workgroup past 2 rounds, 290 -> 319. Up to the measured 512 channels.
bool fused_is_faster(int64_t tiles, int c_in, int c_out, int cus, bool have_uf) {
    if (c_in > 512 || c_out > 512) return false;
    const int64_t items = ceil_div(tiles, kFT) * (c_out / kFC);
    const double fused = 8.0 + double(ceil_div(items, int64_t(cus))) * (6.0 + 3.6 * c_in / kFK) +
                         (have_uf ? 0.0 : 3.0 + double(winograd_fused_bytes(c_out, c_in)) / 1.8e6);
    const double planes = 16.0 * double(tiles);
    const double three = 12.0 + planes * 4.0 * (c_in + c_out) / 4e6 + planes * 2.0 * c_in * c_out / 150e6;
    return fused < three;
}

}  // namespace

size_t winograd_fused_bytes(int c_out, int c_in) { return size_t(16) * c_out * c_in * 6; }

void winograd_fused_weights(Context &ctx, const float *u, int c_out, int c_in, void *uf) {
    MH_REQUIRE(c_in % kFK == 0 && c_out % 32 == 0 && aligned16(u) && aligned16(uf),
               "Winograd fused weights: c_in % 16, c_out % 32, 16-byte aligned");
    const int64_t lanes = int64_t(16) * (c_in / kFK) * (c_out / 32) * 64;
    if (lanes == 0) return;
    const unsigned blocks = unsigned(std::min<int64_t>(ceil_div(lanes, 256), 65536));
    wino_u_fused_kernel<<<blocks, 256, 0, ctx.stream>>>(u, c_out, c_in, static_cast<char *>(uf));
    MH_LAUNCH_CHECK();
}

bool conv3x3_winograd_fused(Context &ctx, const float *x, int n, int h, int w, int c_in, const float *u,
                            const void *uf, int c_out, const float *bias, bool upsample2x, const Affine *prologue,
                            float *out, const float *residual2, GnPartials *gn) {
    if (gn) gn->rows = 0;
    if (ctx.tune.wino_fused == 0 || c_in % 32 || c_out % kFC) return false;
    if (!aligned16(x) || !aligned16(u) || !aligned16(out) || !aligned16(bias) || !aligned16(residual2)) return false;
    if (prologue && (!aligned16(prologue->scale) || !aligned16(prologue->shift))) return false;
    // the kernel's buffer starts a row and a pixel before the input
    const int64_t x_span = (int64_t(n) * h * w + w + 1) * c_in * 4, u_bytes = int64_t(winograd_fused_bytes(c_out, c_in));
    if (x_span > int64_t(kXEnd) || u_bytes >= (int64_t(1) << 31)) return false;
    FGeo g;
    const int up = upsample2x ? 1 : 0;
    g.h = h, g.w = w, g.hi = h << up, g.wi = w << up;
    g.th = (g.hi + 1) / 2, g.tw = (g.wi + 1) / 2;
    const int64_t tiles = int64_t(n) * g.th * g.tw;
    if (ctx.tune.wino_fused < 0 && !fused_is_faster(tiles, c_in, c_out, ctx.cu_count, uf != nullptr)) return false;
    if (tiles == 0) return true;
    g.tiles = int(tiles);
    const int64_t blocks = ceil_div(tiles, kFT) * (c_out / kFC);
    if (blocks >= (int64_t(1) << 30)) return false;
    const int nwork = int(blocks);
    const uint32_t ub = uint32_t(u_bytes);
    if (!uf) {  // no precomputed fused-order copy: make one in the workspace
        void *tmp = ctx.ws.get(size_t(u_bytes), ctx.stream);
        winograd_fused_weights(ctx, u, c_out, c_in, tmp);
        uf = tmp;
    } else if (!aligned16(uf)) {
        return false;
    }
    // GroupNorm partials: blocks of 64 or 32 whole tiles (256 or 128 pixels) within one item
    float *gnp = nullptr;
    const bool halves = int64_t(g.th) * g.tw % kFT != 0;
    if (gn && gn->part && aligned16(gn->part) && g.hi % 2 == 0 && g.wi % 2 == 0 &&
        int64_t(g.th) * g.tw % kHT == 0 && gn->item_rows == g.hi * g.wi) {
        gnp = gn->part;
        gn->rows = 4 * (halves ? kHT : kFT);
    }
    const FArgs a{x,    static_cast<const char *>(uf),
                  prologue ? prologue->scale : nullptr,
                  prologue ? prologue->shift : nullptr,
                  bias, residual2,
                  out,  gnp,
                  ctx.wino_flags, u,
                  g,    ub,
                  c_in, c_out, prologue && prologue->silu ? 1 : 0,
                  c_out / kFC, nwork, halves ? 1 : 0};
    if (up) prologue ? launch_fused<1, true>(ctx, a) : launch_fused<1, false>(ctx, a);
    else prologue ? launch_fused<0, true>(ctx, a) : launch_fused<0, false>(ctx, a);
    MH_LAUNCH_CHECK();
    return true;
}

}  // namespace mh
