// The mean-field level for hidden sizes 16, 32 and 64 on small batches, one workgroup per 16-row tile:
//     h_out = ReLU((A * h_in) * W + bias + msg)
// (examples/graph_classification/src/kernel_mean_field.cpp:37-44) and its backward pass.
//
// On a few thousand rows a level is a chain of latencies: row pointers, entries, gathered rows, contraction, result.  The
// streaming kernel (level_stream.hip) gives a tile to one wavefront, which is right where wavefronts are scarce; here a tile
// has C/16 wavefronts, each of which gathers 16/(C/16) of its rows, one per lane group and up to eight entries of it at
// once, and contracts one 16-column block: a quarter of the gathers and of the matrix instructions in a row at
// C = 64, and W straight into registers (16 values per lane) instead of through LDS.  msg, the gate and the gradient sum do not
// hang on that chain and are asked for ahead of it.  Streaming kernel -> here, us forward and backward:
//     hidden 64, 2.2 entries per row  1,600 rows 5.8 -> 2.9, 6.6 -> 3.8;  7,450 6.1 -> 3.8, 7.3 -> 5.3;  24,576 8.8 -> 7.2, 11.6 -> 11.1
//                30                   1,600      18.6 -> 6.4, 19.6 -> 7.2;  24,576 23.0 -> 16.3, 27.5 -> 21.2
//     hidden 32, 2.2                  1,600      3.6 -> 2.5, 3.9 -> 2.8;  24,576 5.1 -> 4.1, 6.8 -> 6.0;  30: 13.3 -> 9.6, 15.2 -> 12.3
//     hidden 16, 2.2                  1,600      3.3 -> 2.6, 3.5 -> 2.8;  24,576 3.8 -> 3.2, 4.4 -> 4.0;  8: 4.9 -> 4.3, 5.5 -> 5.1
// At 32,000 rows the backward pass at hidden 64 is 12.2 -> 13.6: every workgroup reads W anew, and the result leaves in 64-byte
// pieces of a row; so kLevelTileMaxRows.  At hidden 16 a tile is one wavefront, with nobody to share its gathers: what is left of the
// gain is that they start at once, which long rows outweigh.  With up to 20 entries per row it is as fast as the streaming kernel or faster
// at every number of rows; with 24 to 100 it is, past 12,288 rows, anything from 8 % faster to 13 % slower (30 entries: 14,000 rows
// 7.7 -> 7.9 and 8.1 -> 8.6, 18,000 rows 9.1 -> 8.6 and 9.5 -> 9.2; 100: 20,000 rows 23.9 -> 27.4 and 25.5 -> 29.1), up to there nowhere slower;
// so level_by_tile.  The sums of a row and the products of an element have the order of the streaming kernel, so the bits are the same.
#include "level_gather.h"

namespace gnnhip {
namespace {

// RELU_IN: the gathered rows count as ReLU(row) (the first level reading msg where h0 was not stored)
// BWD: out = (A' x) W^T with the CSR arrays of A' = A^T; A' x is also stored (agg_out), out is zeroed where msg (the gate,
// may be null) is not positive and added to acc_io (may be null); no bias and no ReLU.
template <int C, bool RELU_IN, bool BWD>
__global__ __launch_bounds__(C * 4) void s2v_level_tile_kernel(
    int N, const int* __restrict__ row_ptr, const int* __restrict__ col_idx, const float* __restrict__ val, const float* __restrict__ h_in,
    const float* __restrict__ W, const float* __restrict__ msg, const float* __restrict__ bias, float* __restrict__ h_out,
    float* __restrict__ agg_out, float* __restrict__ acc_io)
{
    constexpr int G = C / 4;             // lanes per gathered row
    constexpr int RPW = kWave / G;       // rows per wavefront, one per lane group
    constexpr int KS = C / 4;            // contraction steps
    constexpr int WAVES = C / 16;        // one per 16-column block
    constexpr int LDT = C + 4;
    constexpr int kRowBytes = C * 4;
    constexpr int kBufEntries = (1 << 30) - 1;                                // entries of col_idx / val a buffer covers
    constexpr int kDirect = G >= 8 ? 8 : 4;                                   // entries per row taken without a loop
    static_assert(RPW * WAVES == 16, "the wavefronts' rows are the tile");

    __shared__ float tile[16 * LDT];
    __shared__ float red_all[WAVES][RPW * C];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int grp = lane / G, tx = lane % G, tx_off = tx * 16;
    const int row0 = (int)blockIdx.x * 16;
    const int lr = wave * RPW + grp, row = row0 + lr;
    float* red = red_all[wave];

    // rows past N read row_ptr[N] twice: no entries
    const int st = row_ptr[min(row, N)], en = row_ptr[min(row + 1, N)];
    // W^T operand of the wavefront's columns: wreg[s] = W[KS q + s][16 wave + t] (BWD: of W transposed)
    float wreg[KS];
    if constexpr (BWD) {
#pragma unroll
        for (int s4 = 0; s4 < KS / 4; ++s4) {
            const float4 v = *reinterpret_cast<const float4*>(W + (size_t)(16 * wave + t) * C + KS * q + 4 * s4);
            wreg[4 * s4 + 0] = v.x; wreg[4 * s4 + 1] = v.y; wreg[4 * s4 + 2] = v.z; wreg[4 * s4 + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int s = 0; s < KS; ++s) wreg[s] = W[(size_t)(KS * q + s) * C + 16 * wave + t];
    }
    // the lane's part of the result: row row0 + t, columns 16 wave + 4 q .. + 3 (a row past N lies outside the buffers)
    const unsigned act_bytes = (unsigned)N * (unsigned)kRowBytes;
    const int out_off = (row0 + t) * kRowBytes + (16 * wave + 4 * q) * 4;
    const rsrc_t msg_rsrc = make_rsrc(msg, msg ? act_bytes : 0u);
    const rsrc_t acc_rsrc = make_rsrc(acc_io, BWD && acc_io ? act_bytes : 0u);
    const float4 mm = buf_load4(msg_rsrc, out_off, 0);
    float4 old = f4_zero(), bias4 = f4_zero();
    if constexpr (BWD) old = buf_load4(acc_rsrc, out_off, 0);
    else if (bias) bias4 = *reinterpret_cast<const float4*>(bias + 16 * wave + 4 * q);

    // the first G entries of the lane group's row, one per lane; rows that are gathered cooperatively take none here
    const rsrc_t ci_rsrc = make_rsrc(col_idx, (unsigned)kBufEntries * 4u);
    const rsrc_t val_rsrc = make_rsrc(val, (unsigned)kBufEntries * 4u);
    const rsrc_t h_rsrc = make_rsrc(h_in, act_bytes);
    const int cnt = en - st;
    const bool together = cnt > kWaveLongRow || (cnt > 0 && en > kBufEntries);
    const bool ok = !together && tx < cnt;
    const int voff = ok ? (st + tx) * 4 : kBufPastEnd;
    const int c0 = buf_load_i(ci_rsrc, voff, 0);
    const float w0 = buf_load_f(val_rsrc, voff, 0);
    const int offs = ok ? c0 * kRowBytes : kBufPastEnd - kRowBytes;           // past the end with tx_off added, too
    float4 x[4], y[4];
    gather4<G, 0>(h_rsrc, offs, tx_off, x);
    if constexpr (kDirect == 8) gather4<G, 4>(h_rsrc, offs, tx_off, y);
    float4 acc = f4_zero();
    sum4<G, 0, RELU_IN>(acc, w0, x);
    if constexpr (kDirect == 8) sum4<G, 4, RELU_IN>(acc, w0, y);
    if (__any(!together && cnt > kDirect)) {
        // the rest of the first batch, then further batches of G
        const int end = together ? st : en;
        for (int base = st; base < end; base += G) {
            int c = c0;
            float v = w0;
            if (base > st) {
                c = 0;
                v = 0.f;
                if (base + tx < end) { c = col_idx[base + tx]; v = val[base + tx]; }
            }
            const int left = min(G, end - base);
            for (int j = base == st ? (kDirect < G ? kDirect : G) : 0; j < left; j += 4) {
                int cj[4];
                float vj[4];
                float4 xx[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) { cj[u] = __shfl(c, (j + u) & (G - 1), G); vj[u] = __shfl(v, (j + u) & (G - 1), G); }
#pragma unroll
                for (int u = 0; u < 4; ++u) xx[u] = buf_load4(h_rsrc, j + u < left ? cj[u] * kRowBytes + tx_off : kBufPastEnd, 0);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (j + u < left) f4_fma(acc, vj[u], as_input<RELU_IN>(xx[u]));
            }
        }
    }
    *reinterpret_cast<float4*>(tile + lr * LDT + tx * 4) = acc;
    // every group of the wavefront takes a share of the entries of each long row
    unsigned long long pending = __ballot(together && tx == 0);
    if (pending) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        while (pending) {
            const int src_lane = __ffsll((long long)pending) - 1;
            pending &= pending - 1;
            const int ls = __shfl(st, src_lane, kWave), le = __shfl(en, src_lane, kWave);
            float4 a = f4_zero();
            int e = ls + grp;
            for (; e + 3 * RPW < le; e += 4 * RPW) {
                int c4[4];
                float v4[4];
                float4 xx[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) { c4[u] = col_idx[e + u * RPW]; v4[u] = val[e + u * RPW]; }
#pragma unroll
                for (int u = 0; u < 4; ++u) xx[u] = buf_load4(h_rsrc, c4[u] * kRowBytes + tx_off, 0);
#pragma unroll
                for (int u = 0; u < 4; ++u) f4_fma(a, v4[u], as_input<RELU_IN>(xx[u]));
            }
            for (; e < le; e += RPW) f4_fma(a, val[e], as_input<RELU_IN>(buf_load4(h_rsrc, col_idx[e] * kRowBytes + tx_off, 0)));
            *reinterpret_cast<float4*>(red + grp * C + tx * 4) = a;
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (grp == src_lane / G) {
                float4 sum = f4_zero();
                for (int g = 0; g < RPW; ++g) {
                    const float4 p = *reinterpret_cast<const float4*>(red + g * C + tx * 4);
                    sum.x += p.x; sum.y += p.y; sum.z += p.z; sum.w += p.w;
                }
                acc = sum;
                *reinterpret_cast<float4*>(tile + lr * LDT + tx * 4) = sum;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    if constexpr (BWD) {
        if (row < N) *reinterpret_cast<float4*>(agg_out + (size_t)row * C + tx * 4) = acc;
    }
    __syncthreads();

    // contraction: lane (q, t) supplies tile[t][KS q + s] at step s and ends with row t, columns 16 wave + 4 q .. + 3
    mfma_f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s4 = 0; s4 < KS / 4; ++s4) {
        const float4 a = *reinterpret_cast<const float4*>(tile + t * LDT + KS * q + 4 * s4);
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[4 * s4 + 0], a.x, sum, 0, 0, 0);
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[4 * s4 + 1], a.y, sum, 0, 0, 0);
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[4 * s4 + 2], a.z, sum, 0, 0, 0);
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[4 * s4 + 3], a.w, sum, 0, 0, 0);
    }
    float4 v = make_float4(sum[0], sum[1], sum[2], sum[3]);
    const rsrc_t out_rsrc = make_rsrc(h_out, act_bytes);
    if constexpr (BWD) {
        if (msg) {
            v.x = mm.x > 0.f ? v.x : 0.f; v.y = mm.y > 0.f ? v.y : 0.f;
            v.z = mm.z > 0.f ? v.z : 0.f; v.w = mm.w > 0.f ? v.w : 0.f;
        }
        // (the buffer is empty where there is no acc_io)
        buf_store4(acc_rsrc, out_off, 0, make_float4(old.x + v.x, old.y + v.y, old.z + v.z, old.w + v.w));
        buf_store4(out_rsrc, out_off, 0, v);
    } else {
        if (bias) { v.x += bias4.x; v.y += bias4.y; v.z += bias4.z; v.w += bias4.w; }
        v.x += mm.x; v.y += mm.y; v.z += mm.z; v.w += mm.w;
        buf_store4(out_rsrc, out_off, 0, relu_ref4(v));
    }
}

template <int C>
int launch_level_tile(int N, const int* row_ptr, const int* col_idx, const float* val, const float* h_in, const float* W, const float* msg,
                      const float* bias, float* h_out, bool relu_in, hipStream_t s)
{
    const dim3 grid((unsigned)(N + 15) / 16), block(C * 4);
    if (relu_in) hipLaunchKernelGGL((s2v_level_tile_kernel<C, true, false>), grid, block, 0, s, N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, (float*)nullptr, (float*)nullptr);
    else hipLaunchKernelGGL((s2v_level_tile_kernel<C, false, false>), grid, block, 0, s, N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, (float*)nullptr, (float*)nullptr);
    GNNHIP_LAUNCH_CHECK("s2v_level_tile");
    return GNNHIP_OK;
}

template <int C>
int launch_level_tile_backward(int N, const int* row_ptr, const int* col_idx, const float* val, const float* x, const float* W,
                               float* agg_out, float* out, const float* gate, float* acc, hipStream_t s)
{
    hipLaunchKernelGGL((s2v_level_tile_kernel<C, false, true>), dim3((unsigned)(N + 15) / 16), dim3(C * 4), 0, s, N, row_ptr, col_idx, val, x, W,
                       gate, (const float*)nullptr, out, agg_out, acc);
    GNNHIP_LAUNCH_CHECK("s2v_level_tile (backward)");
    return GNNHIP_OK;
}

}  // namespace

// N <= kLevelTileMaxRows (level_by_tile); pointers as level_stream_dispatch takes them
int level_tile_dispatch(int N, int C, const int* row_ptr, const int* col_idx, const float* val, const float* h_in, const float* W,
                        const float* msg, const float* bias, float* h_out, bool relu_in, hipStream_t s)
{
    switch (C) {
    case 16: return launch_level_tile<16>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, relu_in, s);
    case 32: return launch_level_tile<32>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, relu_in, s);
    default: return launch_level_tile<64>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, relu_in, s);
    }
}

int level_tile_backward_dispatch(int N, int C, const int* row_ptr, const int* col_idx, const float* val, const float* x, const float* W,
                                 float* agg_out, float* out, const float* gate, float* acc, hipStream_t s)
{
    switch (C) {
    case 16: return launch_level_tile_backward<16>(N, row_ptr, col_idx, val, x, W, agg_out, out, gate, acc, s);
    case 32: return launch_level_tile_backward<32>(N, row_ptr, col_idx, val, x, W, agg_out, out, gate, acc, s);
    default: return launch_level_tile_backward<64>(N, row_ptr, col_idx, val, x, W, agg_out, out, gate, acc, s);
    }
}

}  // namespace gnnhip
