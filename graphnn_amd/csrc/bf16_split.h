// FP32 products on the bf16 matrix cores.
//
// A float x is written as x1 + x2 + x3 with three bf16 numbers: x1 = x rounded to bf16, x2 = the remainder x - x1
// rounded to bf16, x3 what is left.  The remainders are exact in fp32, and the 24 bits of x fit the 3 x 8 bits, so
// the sum of the three is x itself.  A product of two such sums has nine terms; the three smallest (x2 y3, x3 y2,
// x3 y3) are together at most 2^-26 of |x y|, a quarter of what rounding the product once to fp32 costs, and are left
// out.  The other six are exact products of bf16 numbers, which the matrix instruction adds up in fp32: the result
// carries the rounding errors of an fp32 sum and nothing else (measured against float64: no further away than
// v_mfma_f32_16x16x4_f32, whose accumulator is rounded once per four terms instead of once per 32).
//
// Six v_mfma_f32_16x16x32_bf16 cover what takes eight v_mfma_f32_16x16x4_f32: 96 cycles of the matrix pipe instead of
// 256.
//
// Infinities: x1 and x2 are clamped to the largest bf16, so an infinite x leaves its infinity in x3 (no inf - inf), and
// a finite x next to FLT_MAX is not rounded to infinity.  A NaN reaches x3 as well.
#ifndef GNNHIP_BF16_SPLIT_H
#define GNNHIP_BF16_SPLIT_H

#include <hip/hip_runtime.h>

#include "gnnhip_internal.h"

namespace gnnhip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned bf16_words4 __attribute__((ext_vector_type(4)));      // eight bf16 as the registers that hold them

constexpr float kMaxBf16 = 3.3895313892515355e38f;

__device__ __forceinline__ float bf16_clamp(float x) { return __builtin_amdgcn_fmed3f(x, -kMaxBf16, kMaxBf16); }
__device__ __forceinline__ unsigned bf16_pack(float a, float b)         // a in the low half
{
    const bf16x2 p = __builtin_convertvector((float __attribute__((ext_vector_type(2)))){a, b}, bf16x2);
    return __builtin_bit_cast(unsigned, p);
}
__device__ __forceinline__ float bf16_low(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_high(unsigned p) { return __uint_as_float(p & 0xFFFF0000u); }

// the pieces of a and b, packed in pairs: p[i] holds piece i of a in its low half and of b in its high half
__device__ __forceinline__ void bf16_split2(float a, float b, unsigned (&p)[3])
{
    p[0] = bf16_pack(bf16_clamp(a), bf16_clamp(b));
    a -= bf16_low(p[0]); b -= bf16_high(p[0]);
    p[1] = bf16_pack(bf16_clamp(a), bf16_clamp(b));
    a -= bf16_low(p[1]); b -= bf16_high(p[1]);
    p[2] = bf16_pack(a, b);
}

__device__ __forceinline__ mfma_f4 mfma_bf16(const bf16_words4& a, const bf16_words4& b, const mfma_f4& c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace gnnhip

#endif
