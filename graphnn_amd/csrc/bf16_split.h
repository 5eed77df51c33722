// FP32 products on the bf16 matrix cores.
//
// A float x is written as x1 + x2 + x3 with three bf16 numbers: x1 = x rounded to bf16, x2 = the remainder x - x1
// rounded to bf16, x3 what is left.  The remainders are exact in fp32, and the 24 bits of x fit the 3 x 8 bits, so
// the sum of the three is x itself.  A product of two such sums has nine terms; the three smallest (x2 y3, x3 y2,
// x3 y3) are together at most 2^-26 of |x y|, a quarter of what rounding the product once to fp32 costs, and are left
// out.  The other six are exact products of bf16 numbers, which the matrix instruction adds up in fp32.  It rounds
// towards minus infinity, so each kernel sums the corrections (all but x1 y1) ahead of what is large, in the same sum or in one of their own; the
// results are then two to three times closer to float64 than those of v_mfma_f32_16x16x4_f32.
//
// Six v_mfma_f32_16x16x32_bf16 cover what takes eight v_mfma_f32_16x16x4_f32: 96 cycles of the matrix pipe instead of
// 256.
//
// The ends of the range.  The last bits of a number below 2^-110 lie under the smallest bf16, and near the top a correction
// can overflow to the infinity of the other sign.  So operands are scaled before they are split: by 2^16 where everything
// that shares the scale (a row, a column of W, a column over the rows of one workgroup) is below 2^38, which every float down to
// 2^-149 survives whole, and by 2^-63 where something is larger, so that a sum of 256 products of operands scaled either
// way stays finite.  (There, what is below 2^-47 loses its last bits, next to a number of 2^38 or more.  Products of two
// such operands scale back to infinity where they overflow fp32.)  The result is scaled back exactly.  An infinite x is
// split into 1 (with its sign), 0 and the infinity: its product with any y that is not zero has the term x3 y1 of the right
// sign and no other infinite one.  A NaN is a NaN in all its pieces.
#ifndef GNNHIP_BF16_SPLIT_H
#define GNNHIP_BF16_SPLIT_H

#include <hip/hip_runtime.h>

#include "gnnhip_internal.h"

namespace gnnhip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned bf16_words4 __attribute__((ext_vector_type(4)));      // eight bf16 as the registers that hold them

constexpr float kSplitLarge = 0x1p38f;             // from here on an operand is scaled down
constexpr float kSplitUp = 0x1p16f, kSplitUpBack = 0x1p-16f;
constexpr float kSplitDown = 0x1p-63f, kSplitDownBack = 0x1p63f;

// max(m, |a|, |b|), which is what a later m >= kSplitLarge asks about; NaNs are passed over
__device__ __forceinline__ float split_max(float m, float a, float b)
{
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));       // fmaxf would quiet its operands first
    return m;
}

__device__ __forceinline__ unsigned bf16_pack(float a, float b)         // a in the low half
{
    const bf16x2 p = __builtin_convertvector((float __attribute__((ext_vector_type(2)))){a, b}, bf16x2);
    return __builtin_bit_cast(unsigned, p);
}
__device__ __forceinline__ float bf16_low(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_high(unsigned p) { return __uint_as_float(p & 0xFFFF0000u); }

// the pieces of scaled a and b, packed in pairs: p[i] holds piece i of a in its low half and of b in its high half.
// large: they were scaled down, and may be infinite
__device__ __forceinline__ void bf16_split2(float a, float b, bool large, unsigned (&p)[3])
{
    float u = a, v = b;
    if (large) {
        u = isinf(a) ? copysignf(1.f, a) : a;
        v = isinf(b) ? copysignf(1.f, b) : b;
    }
    p[0] = bf16_pack(u, v);
    u -= bf16_low(p[0]); v -= bf16_high(p[0]);
    p[1] = bf16_pack(u, v);
    u -= bf16_low(p[1]); v -= bf16_high(p[1]);
    if (large) {
        u = isinf(a) ? a : u;
        v = isinf(b) ? b : v;
    }
    p[2] = bf16_pack(u, v);
}

__device__ __forceinline__ mfma_f4 mfma_bf16(const bf16_words4& a, const bf16_words4& b, const mfma_f4& c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace gnnhip

#endif
