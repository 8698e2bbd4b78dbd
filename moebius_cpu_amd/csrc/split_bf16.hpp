// f32 values as three bf16 parts, for products on the bf16 matrix instructions
// at f32 precision: x = hi + mid + lo, each part the nearest-even rounding of
// what the parts before it leave, so the three hold all 24 bits of x. A product
// is the sum of the six part products above 2^-24 of it (hi.hi, hi.mid, mid.hi,
// mid.mid, hi.lo, lo.hi), summed in f32. Against the f32 instructions' chain on
// N(0, 1) operands (relative 2-norm error against 64 bits, smallest products
// first): K = 64 1.1e-7 against 1.45e-7, K = 320 2.7e-7 against 3.2e-7, K = 1280
// 5.5e-7 against 6.4e-7, K = 4608 1.07e-6 against 1.21e-6. The bf16 instructions
// issue at 1880 TFLOP/s, so six of them at 313 TFLOP/s against 144 in f32. With the
// five small products in a sum of their own the error is a third of the f32 chain's
// (K = 320 0.8e-7, K = 1280 about 2e-7).
//
// bf16 ends at 2^-133 (its subnormals count), so an operand keeps its 24 bits down to
// 2^-110 and an error of 2^-134 below. That is more than f32 rounding only in sums that
// are small themselves: of a sum s of K products the share is at most 2^-134 times the
// absolute sums of its two operands' K values over s, under 2^-26 while s is at least
// 2^-72 and those sums below 2^36. So the kernels take a sum that is smaller and not
// zero, as one that is infinite or NaN, for one to be redone on the f32 instructions
// (SplitProbe). A sum that is zero because all its operands round to zero (under 2^-134)
// stays zero; with the other side's absolute sum below 2^36 it is under 2^-98. Scaling
// every operand by 2^16 before it is split keeps all bits without that, and cost 1 to
// 3% (UNet step with CFG 6.21 -> 6.40 ms).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mh {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float splitf2 __attribute__((ext_vector_type(2)));

// hi, mid and lo of eight f32 values, each rounded to nearest even.
struct Split3 {
    union Part {
        bf16x2 p[4];
        bf16x8 v;
    } q[3];
};

// What a bf16 part leaves of its value: x - part, exact, as one two-term dot
// product with (-1, 0) or (0, -1) instead of a shift or mask and a subtraction.
// The selectors come through registers: as an inline constant the first would be
// taken for the f32 -1.0, whose bf16 one sits in the upper half.
struct SplitSel {
    bf16x2 e0, e1;
};

__device__ __forceinline__ SplitSel split_sel() {
    uint32_t a = 0x0000bf80u, b = 0xbf800000u;
    asm("" : "+s"(a), "+s"(b));
    return SplitSel{__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b)};
}

__device__ __forceinline__ bf16x2 round_pair(float a, float b) {
    return __builtin_convertvector((splitf2{a, b}), bf16x2);
}

// Pair e of the eight.
__device__ __forceinline__ void split_pair(float a, float b, int e, const SplitSel &sel, Split3 &s) {
    s.q[0].p[e] = round_pair(a, b);
    a = __builtin_amdgcn_fdot2_f32_bf16(s.q[0].p[e], sel.e0, a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(s.q[0].p[e], sel.e1, b, false);
    s.q[1].p[e] = round_pair(a, b);
    a = __builtin_amdgcn_fdot2_f32_bf16(s.q[1].p[e], sel.e0, a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(s.q[1].p[e], sel.e1, b, false);
    s.q[2].p[e] = round_pair(a, b);
}

// The larger magnitude, NaN if either is NaN.
__device__ __forceinline__ float abs_max(float a, float b) {
    return __builtin_elementwise_maximum(__builtin_fabsf(a), __builtin_fabsf(b));
}

// Whether any of the sums seen is infinite, NaN, or too small for its operands' bits.
struct SplitProbe {
    float most = 0.0f;             // the largest magnitude, NaN once a sum is NaN
    uint32_t least = 0xffffffffu;  // the smallest 2 * |bits| - 1: a zero counts as the largest
    __device__ __forceinline__ void see(float a, float b) {
        most = abs_max(abs_max(a, b), most);
        least = min(least, min((__builtin_bit_cast(uint32_t, a) << 1) - 1, (__builtin_bit_cast(uint32_t, b) << 1) - 1));
    }
    __device__ __forceinline__ bool bad() const {
        constexpr uint32_t kLeast = (127u - 72u) << 24;  // 2^-72
        return !(most < __builtin_inff()) || least < kLeast - 1;
    }
};

// Part of a product term t = 0..5 in the order they are summed: {part of A, part of B}.
constexpr int kSplitTerm[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};

}  // namespace
}  // namespace mh
