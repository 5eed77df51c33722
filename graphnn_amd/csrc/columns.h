// How a lane holds the columns of a row of a dense operand: the three packings of the CSR products.
//
// A lane's unit i is the columns i * kVec .. of the row; at(i, n) is the first column it really touches, and
// store_update writes the columns that are the unit's own.  Rows whose width, stride or base is not a multiple of 16 bytes
// are read with 128-bit loads all the same (the hardware wants 4-byte alignment, and a load that straddles two lines
// costs one more access): the row's last unit is moved back to end with the row, so it never reaches past it, and
// repeats up to three columns of the unit before it.  One column per lane instead takes up to four times the lanes, and the
// lanes of a row group past the width are idle (a 300,000-row matrix of 4 entries per row: width 33 in 101 us against 53
// here, width 101 in 140 against 106; a power-law forward at hidden 53, 10 entries per row: 6.9 against 2.9 ms).
#ifndef GNNHIP_COLUMNS_H
#define GNNHIP_COLUMNS_H

#include "gnnhip_internal.h"

namespace gnnhip {

typedef float f32x4_at4 __attribute__((ext_vector_type(4), aligned(4)));

struct ColsWide {                      // 16-byte aligned rows
    static constexpr int kVec = 4;
    using T = float4;
    static __device__ __forceinline__ int at(int unit, int) { return unit * 4; }
    static __device__ __forceinline__ T zero() { return f4_zero(); }
    static __device__ __forceinline__ T load(const float* p) { return *reinterpret_cast<const float4*>(p); }
    static __device__ __forceinline__ void store(float* p, T v) { *reinterpret_cast<float4*>(p) = v; }
    static __device__ __forceinline__ void fma(T& a, float s, T x) { f4_fma(a, s, x); }
    static __device__ __forceinline__ T axpby(T a, float b, T c) { return make_float4(a.x + b * c.x, a.y + b * c.y, a.z + b * c.z, a.w + b * c.w); }
    static __device__ __forceinline__ T add(T a, T b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }
    static __device__ __forceinline__ T relu(T a) { return relu_ref4(a); }
    // row[unit's columns] = v + beta * row[unit's columns]
    static __device__ __forceinline__ void update(float* row, int unit, int, T v, float beta)
    {
        float* p = row + unit * 4;
        store(p, beta == 0.f ? v : axpby(v, beta, load(p)));
    }
};

struct ColsLoose : ColsWide {          // any rows of at least four columns
    static __device__ __forceinline__ int at(int unit, int n) { return min(unit * 4, n - 4); }
    static __device__ __forceinline__ T load(const float* p)
    {
        const f32x4_at4 v = *reinterpret_cast<const f32x4_at4*>(p);
        return make_float4(v.x, v.y, v.z, v.w);
    }
    static __device__ __forceinline__ void store(float* p, T v)
    {
        const f32x4_at4 x = {v.x, v.y, v.z, v.w};
        *reinterpret_cast<f32x4_at4*>(p) = x;
    }
    static __device__ __forceinline__ void update(float* row, int unit, int n, T v, float beta)
    {
        const int c = at(unit, n);
        if (beta == 0.f) {
            store(row + c, v);         // the repeated columns get the same values from both units
            return;
        }
        const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (c + u >= unit * 4) row[c + u] = x[u] + beta * row[c + u];
    }
};

struct ColsOne {                       // fewer than four columns
    static constexpr int kVec = 1;
    using T = float;
    static __device__ __forceinline__ int at(int unit, int) { return unit; }
    static __device__ __forceinline__ T zero() { return 0.f; }
    static __device__ __forceinline__ T load(const float* p) { return *p; }
    static __device__ __forceinline__ void store(float* p, T v) { *p = v; }
    static __device__ __forceinline__ void fma(T& a, float s, T x) { a += s * x; }
    static __device__ __forceinline__ T axpby(T a, float b, T c) { return a + b * c; }
    static __device__ __forceinline__ T add(T a, T b) { return a + b; }
    static __device__ __forceinline__ T relu(T a) { return relu_ref(a); }
    static __device__ __forceinline__ void update(float* row, int unit, int, T v, float beta)
    {
        row[unit] = beta == 0.f ? v : v + beta * row[unit];
    }
};

}  // namespace gnnhip

#endif
