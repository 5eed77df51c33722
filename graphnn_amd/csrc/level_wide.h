// What the kernels of the wide mean-field level (level_wide.hip, level_wide_split.hip) share: batches of CSR entries in
// scalar registers and loads / stores of a lane's part of a row.
#ifndef GNNHIP_LEVEL_WIDE_H
#define GNNHIP_LEVEL_WIDE_H

#include "gnnhip_internal.h"
#include "buffer_addr.h"

namespace gnnhip {
namespace {

constexpr int kInFlight = 6;                     // row gathers in flight per wavefront
constexpr int kWaitVmcnt0 = 0x0F70;              // s_waitcnt operand: vmcnt(0), other counters unconstrained

template <int VEC> struct VecT;
template <> struct VecT<2> { using type = float2; };
template <> struct VecT<4> { using type = float4; };

// Buffer addressing (buffer_addr.h): the memory instruction takes a 128-bit descriptor (base, size), a
// per-lane 32-bit offset and a scalar 32-bit offset, so a gathered row costs one scalar shift and no
// per-lane address arithmetic, and lanes whose offset lies past the size are dropped by the hardware.
template <int VEC> struct BufLoad;
template <> struct BufLoad<4> { static __device__ __forceinline__ float4 get(rsrc_t r, int v, int s) { return buf_load4(r, v, s); } };
template <> struct BufLoad<2> { static __device__ __forceinline__ float2 get(rsrc_t r, int v, int s) { return buf_load2(r, v, s); } };
template <int VEC> struct BufStore;
template <> struct BufStore<4> { static __device__ __forceinline__ void put(rsrc_t r, int v, int s, const float4& x) { buf_store4(r, v, s, x); } };
template <> struct BufStore<2> { static __device__ __forceinline__ void put(rsrc_t r, int v, int s, const float2& x) { buf_store2(r, v, s, x); } };

// A batch of kInFlight consecutive entries of a CSR array (column indices, or edge weights as bit
// patterns) in scalar registers.  The two scalar loads are written as inline assembly with the batch as a
// read-write operand: the loaded values land in the registers the batch already occupies, so a batch that
// is (conditionally) refilled inside the loop needs no copy of the loaded values, and with it no wait for
// the scalar cache right behind the load.  The compiler does not know that these registers are in flight:
// batch_wait() must run before a batch is read.
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
struct Batch { i32x4 lo; i32x2 hi; };
static_assert(kInFlight == 6, "a batch is one 4-dword and one 2-dword scalar load");
__device__ __forceinline__ void batch_load(Batch& b, const int* p)
{
    asm volatile("s_load_dwordx4 %0, %2, 0x0\n\ts_load_dwordx2 %1, %2, 0x10" : "+s"(b.lo), "+s"(b.hi) : "s"(p));
}
// The first n < kInFlight entries of an array that holds no more than n, zeros behind them: one scalar load
// per entry, each under its own (uniform) condition, and the wait right here.
__device__ __forceinline__ void batch_load_short(Batch& b, const int* p, int n)
{
    int t0 = 0, t1 = 0, t2 = 0, t3 = 0, t4 = 0;
    if (n > 0) asm volatile("s_load_dword %0, %1, 0x0" : "+s"(t0) : "s"(p));
    if (n > 1) asm volatile("s_load_dword %0, %1, 0x4" : "+s"(t1) : "s"(p));
    if (n > 2) asm volatile("s_load_dword %0, %1, 0x8" : "+s"(t2) : "s"(p));
    if (n > 3) asm volatile("s_load_dword %0, %1, 0xc" : "+s"(t3) : "s"(p));
    if (n > 4) asm volatile("s_load_dword %0, %1, 0x10" : "+s"(t4) : "s"(p));
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(t0), "+s"(t1), "+s"(t2), "+s"(t3), "+s"(t4));
    b.lo.x = t0; b.lo.y = t1; b.lo.z = t2; b.lo.w = t3;
    b.hi.x = t4; b.hi.y = 0;
}
__device__ __forceinline__ void batch_wait(Batch& b)
{
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(b.lo), "+s"(b.hi));
}
__device__ __forceinline__ int batch_get(const Batch& b, int u)      // u is a compile-time constant after unrolling
{
    return u == 0 ? b.lo.x : u == 1 ? b.lo.y : u == 2 ? b.lo.z : u == 3 ? b.lo.w : u == 4 ? b.hi.x : b.hi.y;
}

template <int VEC, bool RELU_IN>
__device__ __forceinline__ void vec_fma(float (&acc)[VEC], float a, const typename VecT<VEC>::type& x)
{
    const float* p = reinterpret_cast<const float*>(&x);
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = fmaf(a, RELU_IN ? relu_ref(p[i]) : p[i], acc[i]);
}

}  // namespace
}  // namespace gnnhip

#endif
