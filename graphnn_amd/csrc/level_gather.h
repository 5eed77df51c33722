// What the kernels of the narrow mean-field level (level_stream.hip, level_tile.hip) share: gathering the rows of h_in that a
// lane group's row of A names.
#ifndef GNNHIP_LEVEL_GATHER_H
#define GNNHIP_LEVEL_GATHER_H

#include "gnnhip_internal.h"
#include "buffer_addr.h"

namespace gnnhip {

constexpr int kWaveLongRow = 48;     // entries; longer rows are gathered by all groups of the wavefront together,
                                     // and past kHubThreshold they come from the pre-pass when there is one

// Value of lane U of the caller's lane group.  For groups of 16 and of 4 lanes this is a DPP
// operand modifier that the compiler folds into the instruction that consumes the value.
template <int G, int U>
__device__ __forceinline__ int group_lane(int v)
{
    if constexpr (G == 16) return __builtin_amdgcn_mov_dpp(v, 0x150 + U, 0xF, 0xF, true);          // row_newbcast:U
    else if constexpr (G == 4) return __builtin_amdgcn_mov_dpp(v, U * 0x55, 0xF, 0xF, true);        // quad_perm:[U,U,U,U]
    else return __shfl(v, U, G);
}
template <int G, int U>
__device__ __forceinline__ float group_lane(float v)
{
    return __int_as_float(group_lane<G, U>(__float_as_int(v)));
}

// x[u] = h_in[entry U0 + u of the lane group's row], u = 0..3: offs holds, per lane of the group, the byte
// offset of the entry's row of h_in (past the end where the row has no such entry: the load reads zeros)
template <int G, int U0>
__device__ __forceinline__ void gather4(rsrc_t h_rsrc, int offs, int tx_off, float4 (&x)[4])
{
    x[0] = buf_load4(h_rsrc, group_lane<G, U0 + 0>(offs) + tx_off, 0);
    x[1] = buf_load4(h_rsrc, group_lane<G, U0 + 1>(offs) + tx_off, 0);
    x[2] = buf_load4(h_rsrc, group_lane<G, U0 + 2>(offs) + tx_off, 0);
    x[3] = buf_load4(h_rsrc, group_lane<G, U0 + 3>(offs) + tx_off, 0);
}
// RELU_IN: the gathered rows count as ReLU(row) (the first level reading msg where h0 was not stored)
template <bool RELU_IN>
__device__ __forceinline__ float4 as_input(const float4& x)
{
    return RELU_IN ? relu_ref4(x) : x;
}
template <int G, int U0, bool RELU_IN>
__device__ __forceinline__ void sum4(float4& acc, float w, const float4 (&x)[4])
{
    f4_fma(acc, group_lane<G, U0 + 0>(w), as_input<RELU_IN>(x[0]));
    f4_fma(acc, group_lane<G, U0 + 1>(w), as_input<RELU_IN>(x[1]));
    f4_fma(acc, group_lane<G, U0 + 2>(w), as_input<RELU_IN>(x[2]));
    f4_fma(acc, group_lane<G, U0 + 3>(w), as_input<RELU_IN>(x[3]));
}

}  // namespace gnnhip

#endif
