// Input stage for hidden sizes 128 and 256 (and 64 when only msg is wanted) and up to 64 label types:
//     msg = X * W_n2l ,  h0 = ReLU(msg)
// MatMul + ReLU of examples/graph_classification/src/kernel_mean_field.cpp:31-32 in one pass,
// with the K x C contraction on the FP32 matrix cores.
//
// A workgroup of four wavefronts takes 64 rows of X at a time into LDS (zero-padded to a
// multiple of four columns); wavefront w owns the output columns [w C/4, (w+1) C/4) and keeps
// its slice of W_n2l^T in registers for the whole launch.  Operand roles are swapped
// (out^T = W^T * X^T) so that a lane ends up with four consecutive output columns of one row:
// 128-bit stores of msg and of h0.  msg and h0 are addressed through buffer descriptors that
// cover the rows of the current tile only, so rows past N need no predicate.
//
// Algorithmic bytes: 4 N (K + 2 C) + 4 K C; flops 2 N K C.  HBM-bound (the two outputs).
#include "bf16_split.h"
#include "buffer_addr.h"

namespace gnnhip {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;       // 4
constexpr int kTileRows = 64;

// KS = contraction steps of four: K <= 4 KS.  PIECES: products from bf16 pieces (bf16_split.h).  ROWS: a wavefront forms 16 whole rows, which leave
// through LDS row by row
template <int C, int KS, bool GATED, bool PIECES, bool ROWS>
__global__ __launch_bounds__(kBlock) void s2v_input_wide_kernel(
    int N, int K, unsigned k_magic, int x_vec, const float* __restrict__ X, const float* __restrict__ Wn2l,
    float* __restrict__ msg, float* __restrict__ h0, const int* __restrict__ gate)
{
    if (gated_off<GATED>(gate)) return;
    constexpr int CW = ROWS ? C : C / kWaves;                // output columns per wavefront
    constexpr int NB = CW / 16;              // 16-column blocks per wavefront
    constexpr int LDT = 4 * KS + 4;          // LDS row stride
    constexpr int KS2 = (KS + 7) / 8;        // contraction steps in pieces
    __shared__ float xt[kTileRows * LDT];
    __shared__ float w_down[PIECES ? C : 1]; // a column's scale up over its scale
    __shared__ float out_all[ROWS ? kWaves * 16 * (C + 4) : 1];

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int q = lane >> 4, t = lane & 15;
    const int col0 = ROWS ? 0 : wave * CW;

    // W^T operand: wreg[jb][s] = W_n2l[KS q + s][col0 + 16 jb + t], zero past K; in pieces: of W_n2l[KS q + 8 s + 0..7].  The matrix
    // instructions on bf16 round towards minus infinity: every other block of columns is formed with -W
    float wreg[PIECES ? 1 : NB][PIECES ? 1 : KS];
    bf16_words4 wp[PIECES ? NB : 1][PIECES ? KS2 : 1][3];
    bool any_down = false;                   // a column is scaled down: uniform
    auto w_at = [&](int jb, int s) { return KS * q + s < K ? Wn2l[(size_t)(KS * q + s) * C + col0 + 16 * jb + t] : 0.f; };
    if constexpr (PIECES) {
        static_assert(KS == 8 * KS2, "whole steps");
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) {
            float w[KS], largest = 0.f;
#pragma unroll
            for (int s = 0; s < KS; ++s) w[s] = w_at(jb, s);
#pragma unroll
            for (int s = 0; s < KS; s += 2) largest = split_max(largest, w[s], w[s + 1]);
            const unsigned long long large = __ballot(largest >= kSplitLarge);
            const bool down = (large >> t) & 0x0001000100010001ull;              // in any quarter of the column
            any_down |= large != 0;
            const float scale = down ? kSplitDown : kSplitUp;
            if (q == 0) w_down[col0 + 16 * jb + t] = down ? kSplitUp / kSplitDown : 1.f;
#pragma unroll
            for (int s = 0; s < KS2; ++s)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    unsigned p[3];
                    bf16_split2(w[8 * s + 2 * u] * scale, w[8 * s + 2 * u + 1] * scale, down, p);
#pragma unroll
                    for (int n = 0; n < 3; ++n) wp[jb][s][n][u] = p[n] ^ (jb % 2 ? 0x80008000u : 0u);
                }
        }
    } else {
#pragma unroll
        for (int jb = 0; jb < NB; ++jb)
#pragma unroll
            for (int s = 0; s < KS; ++s) wreg[jb][s] = w_at(jb, s);
    }

    const int lane_off = (t * C + col0 + 4 * q) * 4;      // byte offset of this lane inside a 16-row block
    const int ntiles = (int)(((long long)N + kTileRows - 1) / kTileRows);
    // X rows of a tile, asked for before the contraction of the previous tile.  A full tile is 64 K
    // contiguous floats: with x_vec set (X 16-byte aligned) the workgroup reads them as KS/4 128-bit words per
    // lane and scatters them into the padded LDS rows (row = element / K by one multiply-high with
    // ceil(2^32 / K)); the last, partial tile and unaligned X go row by row: wavefront w copies rows
    // 16 w .. 16 w + 15, one row per load.
    constexpr int XQ = KS / 4;
    float xv[16];
    float4 xq[XQ];
    for (int i = threadIdx.x; i < kTileRows * LDT; i += kBlock) xt[i] = 0.f;      // the padding columns stay zero
    auto full_tile = [&](int tile) { return x_vec && (long long)(tile + 1) * kTileRows <= (long long)N; };
    auto load_x = [&](int tile) {
        if (full_tile(tile)) {
            const float4* xg = reinterpret_cast<const float4*>(X + (size_t)tile * kTileRows * K);
#pragma unroll
            for (int p = 0; p < XQ; ++p) {
                const int f = threadIdx.x + p * kBlock;
                xq[p] = (f * 4 < kTileRows * K) ? xg[f] : f4_zero();
            }
        } else {
            const long long r0 = (long long)tile * kTileRows + wave * 16;
#pragma unroll
            for (int rr = 0; rr < 16; ++rr)
                xv[rr] = (lane < K && r0 + rr < N) ? X[(size_t)(r0 + rr) * K + lane] : 0.f;
        }
    };
    auto park_x = [&](int tile) {
        if (full_tile(tile)) {
#pragma unroll
            for (int p = 0; p < XQ; ++p) {
                const int e = (threadIdx.x + p * kBlock) * 4;
                if (e < kTileRows * K) {
                    int r = K >= 2 ? (int)__umulhi((unsigned)e, k_magic) : e;
                    int c = e - r * K;
                    const float v[4] = {xq[p].x, xq[p].y, xq[p].z, xq[p].w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        xt[r * LDT + c] = v[i];           // 64 K is a multiple of 4: the four elements exist
                        if (++c == K) { c = 0; ++r; }
                    }
                }
            }
        } else {
#pragma unroll
            for (int rr = 0; rr < 16; ++rr)
                if (lane < 4 * KS) xt[(wave * 16 + rr) * LDT + lane] = xv[rr];
        }
    };
    if ((int)blockIdx.x < ntiles) load_x(blockIdx.x);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const long long row0 = (long long)tile * kTileRows;
        const long long left = (long long)N - row0;
        const int rows = (int)(left < kTileRows ? left : kTileRows);
        __syncthreads();                     // the previous tile has been consumed (first pass: the zero fill is done)
        park_x(tile);
        __syncthreads();
        if (tile + (int)gridDim.x < ntiles) load_x(tile + gridDim.x);

        const unsigned bytes = (unsigned)rows * (C * 4);
        const rsrc_t msg_rsrc = make_rsrc(msg + (size_t)row0 * C, bytes);
        const rsrc_t h0_rsrc = make_rsrc(h0 ? h0 + (size_t)row0 * C : nullptr, h0 ? bytes : 0u);      // h0 may be null
#pragma unroll 1
        for (int rt = ROWS ? __builtin_amdgcn_readfirstlane(wave) : 0; rt < (ROWS ? __builtin_amdgcn_readfirstlane(wave) + 1 : kTileRows / 16); ++rt) {
            if (rt * 16 >= rows) break;
            mfma_f4 acc[NB];
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) acc[jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};
            const float* src = xt + (rt * 16 + t) * LDT + KS * q;
            float back = 1.f;
            if constexpr (PIECES) {
                float x[KS], largest = 0.f;
#pragma unroll
                for (int s = 0; s < KS; s += 4) {
                    const float4 b = *reinterpret_cast<const float4*>(src + s);
                    x[s] = b.x; x[s + 1] = b.y; x[s + 2] = b.z; x[s + 3] = b.w;
                }
#pragma unroll
                for (int s = 0; s < KS; s += 2) largest = split_max(largest, x[s], x[s + 1]);
                const unsigned long long large = __ballot(largest >= kSplitLarge);
                bf16_words4 p[KS2][3];
                auto split = [&](float scale, bool down) {
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            unsigned w[3];
                            bf16_split2(x[8 * s + 2 * u] * scale, x[8 * s + 2 * u + 1] * scale, down, w);
                            p[s][0][u] = w[0]; p[s][1][u] = w[1]; p[s][2][u] = w[2];
                        }
                };
                back = kSplitUpBack * kSplitUpBack;
                if (large) {                 // uniform: some row is scaled down
                    const bool down = (large >> t) & 0x0001000100010001ull;
                    split(down ? kSplitDown : kSplitUp, down);
                    if (down) back = kSplitDownBack * kSplitUpBack;
                } else {
                    split(kSplitUp, false);
                }
                // the corrections first, in the same sum
                auto products = [&](int w, int n) {
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NB; ++jb) acc[jb] = mfma_bf16(wp[jb][s][w], p[s][n], acc[jb]);
                };
                products(2, 0); products(0, 2); products(1, 1); products(1, 0); products(0, 1); products(0, 0);
            } else {
#pragma unroll
                for (int s4 = 0; s4 < KS / 4; ++s4) {
                    const float4 b = *reinterpret_cast<const float4*>(src + 4 * s4);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][4 * s4 + 0], b.x, acc[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][4 * s4 + 1], b.y, acc[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][4 * s4 + 2], b.z, acc[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][4 * s4 + 3], b.w, acc[jb], 0, 0, 0);
                }
            }
            const int voff = lane_off + rt * (16 * C * 4);
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                float4 v = make_float4(acc[jb][0], acc[jb][1], acc[jb][2], acc[jb][3]);
                if constexpr (PIECES) {
                    const float b = jb % 2 ? -back : back;
                    float4 f = make_float4(b, b, b, b);
                    if (any_down) {
                        const float4 d = *reinterpret_cast<const float4*>(w_down + col0 + 16 * jb + 4 * q);
                        f.x *= d.x; f.y *= d.y; f.z *= d.z; f.w *= d.w;
                    }
                    v = make_float4(fmaf(v.x, f.x, 0.f), fmaf(v.y, f.y, 0.f), fmaf(v.z, f.z, 0.f), fmaf(v.w, f.w, 0.f));     // no -0 for 0
                }
                if constexpr (ROWS) {
                    *reinterpret_cast<float4*>(out_all + (wave * 16 + t) * (C + 4) + 16 * jb + 4 * q) = v;
                } else {
                    buf_store4(msg_rsrc, voff + 64 * jb, 0, v);
                    if (h0) buf_store4(h0_rsrc, voff + 64 * jb, 0, relu_ref4(v));
                }
            }
            if constexpr (ROWS) {
                constexpr int kLanes = C / 4, kTogether = kWave / kLanes;        // lanes of a row, rows of a store
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
                for (int r0 = 0; r0 < 16; r0 += kTogether) {
                    const int r = r0 + lane / kLanes, c = 4 * (lane % kLanes);
                    const float4 v = *reinterpret_cast<const float4*>(out_all + (wave * 16 + r) * (C + 4) + c);
                    buf_store4(msg_rsrc, ((rt * 16 + r) * C + c) * 4, 0, v);
                    if (h0) buf_store4(h0_rsrc, ((rt * 16 + r) * C + c) * 4, 0, relu_ref4(v));
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            }
        }
    }
}

template <int C, int KS>
int launch_input_wide(int N, int K, const float* X, const float* Wn2l, float* msg, float* h0, hipStream_t s, const int* gate)
{
    const long long ntiles = ((long long)N + kTileRows - 1) / kTileRows;
    // What bounds the large calls is how the outputs reach memory.  Past what the memory-side cache holds (256 MB of outputs), fewer rows in the
    // writing at once are faster (hidden 128 with h0, K = 7: 300,000 rows 67 us with four workgroups per compute unit, 63 with two,
    // 700,000 171 and 135; hidden 256 without, K = 32: 300,000 rows 88 and 79; six or eight are slower than four), and so are whole rows per store
    // where W's operand for all columns is small (hidden 64 without h0, K = 16: 2,500,000 rows 176 -> 148, 60,000 6.2 -> 6.6; 128, K = 16: 700,000
    // 98 -> 76); at hidden 256 with h0 fewer in the writing gain from 400 MB on (K = 32: 180,000 rows 89.7 and 93.3, 250,000 133.7 and 129.7).
    // At hidden 256 and K > 32 two workgroups leave room for their registers (K = 48: 60,000 rows 22.8 -> 19.6, 90,000 28.4 -> 26.4; K = 64
    // with h0 45,000 26.3 -> 23.4, 90,000 45.9 -> 41.8), but up to three tiles per compute unit at K <= 48 (45,000 15.9 and 16.5), and for K > 48 with h0 past
    // what the cache holds (180,000 93.6 and 97.3, 300,000 150.6 and 153.6).
    // K > 48, hidden 256, msg alone: the FP32 matrix instructions, and all that waits for a slot between them, are longer
    // than the outputs (300,000 rows 109 us, K = 4 63); in pieces 85.  Hidden 128, and with h0, gain nothing from that, nor do up to two tiles per compute
    // unit, which wait for W to be split (2,000 rows 8.7 us and 10.7 in pieces, 16,000 10.2 and 12.3, 30,000 14.7 and 15.5, 33,000 22.2 and 18.4).
    const unsigned long long out_bytes = (h0 ? 2ull : 1ull) * (unsigned long long)N * C * 4ull;
    const bool big = out_bytes > (256ull << 20);
    const bool pieces = C == 256 && KS == 16 && !h0 && ntiles > 2 * kNumCU, rows = big && !h0 && (C == 64 ? KS <= 8 : C == 128 && KS == 4);
    const bool two = C == 256 && KS == 12 ? ntiles > 3 * kNumCU : C == 256 && KS == 16 ? (h0 ? !big : pieces) :
                     C >= 128 && out_bytes > ((C == 256 && h0 ? 400ull : 256ull) << 20) && (h0 || KS < 16) && !rows;
    const long long cap = (long long)kNumCU * (two ? 2 : 4);
    const unsigned grid = (unsigned)(ntiles < cap ? ntiles : cap);
    const unsigned k_magic = K >= 2 ? (unsigned)((0x100000000ull + (unsigned)K - 1) / (unsigned)K) : 0u;   // ceil(2^32 / K)
    const int x_vec = aligned16(X) ? 1 : 0;
    constexpr bool kGated = C == 64;             // the size of batch_forward.hip among these
    auto kernel = kGated && gate ? &s2v_input_wide_kernel<C, KS, kGated, false, false> : &s2v_input_wide_kernel<C, KS, false, false, false>;
    if constexpr (C == 256 && KS == 16) {
        if (pieces) kernel = &s2v_input_wide_kernel<C, KS, false, true, false>;
    } else if constexpr ((C == 64 && KS <= 8) || (C == 128 && KS == 4)) {
        if (rows) kernel = kGated && gate ? &s2v_input_wide_kernel<C, KS, kGated, false, true> : &s2v_input_wide_kernel<C, KS, false, false, true>;
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, s, N, K, k_magic, x_vec, X, Wn2l, msg, h0, gate);
    GNNHIP_LAUNCH_CHECK("s2v_input_wide");
    return GNNHIP_OK;
}

template <int C>
int input_wide_c(int N, int K, const float* X, const float* Wn2l, float* msg, float* h0, hipStream_t s, const int* gate)
{
    if (K <= 16) return launch_input_wide<C, 4>(N, K, X, Wn2l, msg, h0, s, gate);
    if (K <= 32) return launch_input_wide<C, 8>(N, K, X, Wn2l, msg, h0, s, gate);
    if (K <= 48) return launch_input_wide<C, 12>(N, K, X, Wn2l, msg, h0, s, gate);
    return launch_input_wide<C, 16>(N, K, X, Wn2l, msg, h0, s, gate);
}

}  // namespace

int input_wide_dispatch(int N, int K, int C, const float* X, const float* Wn2l, float* msg, float* h0, hipStream_t s, const int* gate)
{
    if (K > 64 || !(aligned16(msg) && aligned16(h0))) return GNNHIP_EUNSUPPORTED;
    switch (C) {
    case 64: return input_wide_c<64>(N, K, X, Wn2l, msg, h0, s, gate);
    case 128: return input_wide_c<128>(N, K, X, Wn2l, msg, h0, s, gate);
    case 256: return input_wide_c<256>(N, K, X, Wn2l, msg, h0, s, gate);
    }
    return GNNHIP_EUNSUPPORTED;
}

}  // namespace gnnhip
