// Readout of batches of many small graphs, one wavefront per graph:
//     pool = S * h ; hidden = ReLU(pool * W_h1) ; logits = hidden * W_h2 ;
//     probs = softmax(logits) ; pred = argmax(logits)
// (MatMul(S, h) -> MatMul -> ReLU -> MatMul of examples/graph_classification/src/kernel_mean_field.cpp:45-49,
// row softmax of src/tensor/gpu_dense_tensor.cu:298-370, arg-max with the lowest index winning ties as in
// src/tensor/cpu_dense_tensor.cpp:176-196.)
//
// W_h1 and W_h2 are copied into LDS once per workgroup.  A wavefront then takes graphs g, g + nwaves, ...
// and never synchronises with the other wavefronts of its workgroup:
//   1. sum-pool: G = C/4 lanes take one row of h as float4s; the 64/G lane groups walk the graph's rows
//      four at a time each, their sums are added in group order through LDS;
//   2. hidden: lane j adds pool[c] * W_h1[c][j] over c in order (pool broadcast from LDS, W_h1 rows read by
//      consecutive lanes);
//   3. logits the same way over the hidden units, then softmax and arg-max inside the wavefront.
// Hidden sizes 16, 32 and 64 (at 256 the weights fill LDS, one workgroup per CU remains, and SpMM + GEMM
// are faster: 140 against 204 us for 10,000 graphs).  Algorithmic bytes: 4NC (h) + 8N (S) + 4B(C + H + 2Q) + 4(CH + HQ).
#include "columns.h"
#include <math.h>
#include <type_traits>

namespace gnnhip {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kMaxLds = 150 * 1024;

// POOL: the pooled rows alone, of a gated launch
template <int C, bool POOL>
__global__ __launch_bounds__(kBlock) void s2v_readout_wave_kernel(
    int B, int H, int Q, const int* __restrict__ s_row_ptr, const int* __restrict__ s_col_idx,
    const float* __restrict__ s_val, const float* __restrict__ h, const float* __restrict__ Wh1,
    const float* __restrict__ Wh2, float* __restrict__ pool, float* __restrict__ hidden,
    float* __restrict__ logits, float* __restrict__ probs, int* __restrict__ pred, const int* __restrict__ gate)
{
    if (gated_off<POOL>(gate)) return;
    constexpr int G = C / 4;             // lanes per row of h
    constexpr int RPR = kWave / G;       // rows in flight per step of the wavefront
    extern __shared__ float smem[];
    float* w1 = smem;                    // [C][H]
    float* w2 = w1 + (size_t)C * H;      // [H][Q]
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int per_wave = RPR * C + C + H + Q;
    float* part = w2 + (size_t)H * Q + (size_t)wave * per_wave;   // [RPR][C]
    float* pl = part + RPR * C;          // [C]
    float* hid = pl + C;                 // [H]
    float* lg = hid + H;                 // [Q]
    const int grp = lane / G, tx = lane % G;

    if constexpr (!POOL) {
        for (int i = threadIdx.x; i < C * H; i += kBlock) w1[i] = Wh1[i];
        for (int i = threadIdx.x; i < H * Q; i += kBlock) w2[i] = Wh2[i];
        __syncthreads();
    }

    const int nwaves = (int)gridDim.x * kWavesPerBlock;
    for (int g = (int)blockIdx.x * kWavesPerBlock + wave; g < B; g += nwaves) {
        const int start = s_row_ptr[g], end = s_row_ptr[g + 1];
        // ---- sum-pool
        float4 acc = f4_zero();
        int t = start + grp;
        for (; t + 3 * RPR < end; t += 4 * RPR) {
            int c[4];
            float v[4];
            float4 x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { c[u] = s_col_idx[t + u * RPR]; v[u] = s_val[t + u * RPR]; }
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const float4*>(h + (size_t)c[u] * C + tx * 4);
#pragma unroll
            for (int u = 0; u < 4; ++u) f4_fma(acc, v[u], x[u]);
        }
        for (; t < end; t += RPR)
            f4_fma(acc, s_val[t], *reinterpret_cast<const float4*>(h + (size_t)s_col_idx[t] * C + tx * 4));
        *reinterpret_cast<float4*>(part + grp * C + tx * 4) = acc;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        for (int cc = lane; cc < C; cc += kWave) {
            float s = 0.f;
#pragma unroll
            for (int p = 0; p < RPR; ++p) s += part[p * C + cc];
            pl[cc] = s;
            pool[(size_t)g * C + cc] = s;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if constexpr (POOL) continue;
        // ---- hidden = ReLU(pool * W_h1)
        for (int j = lane; j < H; j += kWave) {
            float s = 0.f;
#pragma unroll 16
            for (int cc = 0; cc < C; ++cc) s += pl[cc] * w1[(size_t)cc * H + j];
            s = relu_ref(s);
            hid[j] = s;
            hidden[(size_t)g * H + j] = s;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        // ---- logits = hidden * W_h2
        for (int q = lane; q < Q; q += kWave) {
            float s = 0.f;
#pragma unroll 8
            for (int j = 0; j < H; ++j) s += hid[j] * w2[(size_t)j * Q + q];
            lg[q] = s;
            logits[(size_t)g * Q + q] = s;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        // ---- softmax + argmax over Q
        if (probs || pred) {
            const float first = lg[0];
            float mx = first;                       // the reference scan starts at element 0
            float bv = -INFINITY;
            int bi = 0x7fffffff;
            for (int q = lane; q < Q; q += kWave) {
                const float v = lg[q];
                mx = max_keep(mx, v);
                const float vv = (v != v) ? -INFINITY : v;     // a NaN that is not first never wins
                argmax_combine(bv, bi, vv, q);
            }
            mx = wave_max(mx);
            wave_argmax(bv, bi);
            if (first != first) bi = 0;             // a NaN in column 0 is never displaced
            if (pred && lane == 0) pred[g] = bi;
            if (probs) {
                float s = 0.f;
                for (int q = lane; q < Q; q += kWave) {
                    const float e = expf(lg[q] - mx);
                    lg[q] = e;
                    s += e;
                }
                s = wave_sum(s);
                for (int q = lane; q < Q; q += kWave) probs[(size_t)g * Q + q] = lg[q] / s;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");     // the wavefront's LDS rows are reused by its next graph
    }
}

template <int C, bool POOL = false>
int launch_readout_wave(int B, int H, int Q, const int* s_row_ptr, const int* s_col_idx, const float* s_val,
                        const float* h, const float* Wh1, const float* Wh2, float* pool, float* hidden,
                        float* logits, float* probs, int* pred, hipStream_t s, const int* gate = nullptr)
{
    constexpr int RPR = kWave / (C / 4);
    const size_t smem = sizeof(float) * ((size_t)C * H + (size_t)H * Q + (size_t)kWavesPerBlock * (RPR * C + C + H + Q));
    if (smem > (size_t)kMaxLds) return GNNHIP_EUNSUPPORTED;
    auto kernel = s2v_readout_wave_kernel<C, POOL>;
    static LdsLimit lds_limit;               // one per kernel instantiation
    GNNHIP_HIP(lds_limit.raise(reinterpret_cast<const void*>(kernel), smem > 64 * 1024 ? (size_t)kMaxLds : smem));
    const long long blocks_needed = ((long long)B + kWavesPerBlock - 1) / kWavesPerBlock;
    const long long per_cu = smem > 0 ? (long long)(160 * 1024) / (long long)smem : 8;
    long long cap = (long long)kNumCU * (per_cu < 1 ? 1 : (per_cu > 8 ? 8 : per_cu));
    const unsigned grid = (unsigned)(blocks_needed < cap ? blocks_needed : cap);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), smem, s, B, H, Q, s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2,
                       pool, hidden, logits, probs, pred, gate);
    GNNHIP_LAUNCH_CHECK("s2v_readout_wave");
    return GNNHIP_OK;
}

// Readout for wide hidden sizes (C = 128 or 256) on batches of thousands of graphs: one workgroup per tile of
// kTileGraphs graphs.  W_h1 (128 KB at 256 x 128) does not fit LDS next to anything else, so it stays in memory
// and every tile streams it once through L2:
//   1. sum-pool   a wavefront per graph, the whole wavefront across the C columns of a row, rows in order
//                 (the order of the reference path), eight loads in flight; pooled rows go to LDS [graphs][C].  A graph is a
//                 chain of trips, so what bounds this is how many are summed at once: four wavefronts per tile, four graphs each in turn,
//                 were 76 us at 10,000 graphs of 30 nodes, hidden 256, sixteen are 71, where a copy of the rows' bytes takes 59;
//   2. hidden     on the FP32 matrix cores, a wavefront per 16 units (10,000 graphs of 30 nodes, hidden 256, 128 units: 92 -> 83 us; a lane per
//                 unit and eight graphs, with the pooled rows broadcast from LDS, was a tenth of the launch);
//   3. logits     a lane per (graph, class), the sum over the hidden units in order;
//   4. softmax and arg-max inside a wavefront per graph, as in the kernel above.
// Algorithmic bytes as above; W_h1 traffic from L2 is 4 C H per tile.
constexpr int kTileGraphs = 16;

template <int C, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void s2v_readout_tile_kernel(
    int B, int H, int Q, const int* __restrict__ s_row_ptr, const int* __restrict__ s_col_idx,
    const float* __restrict__ s_val, const float* __restrict__ h, const float* __restrict__ Wh1,
    const float* __restrict__ Wh2, float* __restrict__ pool, float* __restrict__ hidden,
    float* __restrict__ logits, float* __restrict__ probs, int* __restrict__ pred)
{
    constexpr int VEC = C / kWave;       // floats of a row per lane (2 or 4)
    constexpr int kAhead = 16;
    constexpr int LD = C + 4;
    using vec_t = typename std::conditional<VEC == 4, float4, float2>::type;
    extern __shared__ float smem[];
    float* pl = smem;                                // [kTileGraphs][LD]
    float* hid = pl + kTileGraphs * LD;              // [kTileGraphs][H]
    float* lg = hid + (size_t)kTileGraphs * H;       // [kTileGraphs][Q]
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int g0 = (int)blockIdx.x * kTileGraphs;
    const int ng = min(kTileGraphs, B - g0);

    // ---- sum-pool: the offsets of all graphs in one trip, the first 64 node indices and weights of a graph on their way while the one
    //      before it is summed, handed round lane by lane; eight rows in flight, added in row order
    const int offsets = s_row_ptr[g0 + min(lane, ng)];
    auto offset = [&](int gi) { return __builtin_amdgcn_readlane(offsets, min(gi, ng)); };
    int next_c = 0;
    float next_v = 0.f;
    auto ask = [&](int gi) {
        const int e = offset(gi) + lane;
        if (e < offset(gi + 1)) { next_c = s_col_idx[e]; next_v = s_val[e]; }
    };
    ask(wave);
    for (int gi = wave; gi < kTileGraphs; gi += WAVES) {
        float acc[VEC];
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
        const int start = offset(gi), end = offset(gi + 1);      // the same past the last graph
        int my_c = next_c;
        float my_v = next_v;
        if (gi + WAVES < kTileGraphs) ask(gi + WAVES);
        for (int base = start; base < end; base += kWave) {
            const int cnt = min(kWave, end - base);
            if (base > start && lane < cnt) { my_c = s_col_idx[base + lane]; my_v = s_val[base + lane]; }
            for (int j = 0; j < cnt; j += 8) {
                vec_t x[8];
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int src = min(j + u, cnt - 1);                     // uniform
                    const int c = __builtin_amdgcn_readlane(my_c, src);
                    v[u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_v), src));
                    x[u] = *reinterpret_cast<const vec_t*>(h + (size_t)c * C + lane * VEC);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    if (j + u < cnt) {
                        const float* xp = reinterpret_cast<const float*>(&x[u]);
#pragma unroll
                        for (int i = 0; i < VEC; ++i) acc[i] = fmaf(v[u], xp[i], acc[i]);
                    }
                }
            }
        }
        if (gi < ng) *reinterpret_cast<vec_t*>(pool + (size_t)(g0 + gi) * C + lane * VEC) = *reinterpret_cast<vec_t*>(acc);
        *reinterpret_cast<vec_t*>(pl + gi * LD + lane * VEC) = *reinterpret_cast<vec_t*>(acc);   // zeros past the last graph
    }
    __syncthreads();

    // ---- hidden = ReLU(pool * W_h1): a wavefront per 16 units, whose operand comes straight from memory, 16 contraction steps ahead; lane
    //      (q, t) takes columns KS q .. KS q + KS - 1 of graph t and ends up with units 4 q .. of it
    constexpr int KS = C / 4;
    const int q4 = lane >> 4, t = lane & 15;
    for (int j0 = 16 * wave; j0 < H; j0 += 16 * WAVES) {
        const float* w1 = Wh1 + (size_t)(KS * q4) * H + min(j0 + t, H - 1);
        const float* x = pl + t * LD + KS * q4;
        float w[2][kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; ++s) w[0][s] = w1[(size_t)s * H];
        mfma_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s0 = 0; s0 < KS; s0 += kAhead) {
            const int cur = s0 / kAhead % 2;
            if (s0 + kAhead < KS) {
#pragma unroll
                for (int s = 0; s < kAhead; ++s) w[cur ^ 1][s] = w1[(size_t)(s0 + kAhead + s) * H];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < kAhead; s += 4) {
                const float4 v = *reinterpret_cast<const float4*>(x + s0 + s);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[cur][s], v.x, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[cur][s + 1], v.y, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[cur][s + 2], v.z, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[cur][s + 3], v.w, acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = j0 + 4 * q4 + i;
            if (j >= H) continue;
            const float v = relu_ref(acc[i]);
            hid[(size_t)t * H + j] = v;
            if (t < ng) hidden[(size_t)(g0 + t) * H + j] = v;
        }
    }
    __syncthreads();

    // ---- logits = hidden * W_h2
    for (int it = threadIdx.x; it < kTileGraphs * Q; it += WAVES * kWave) {
        const int gi = it / Q, q = it % Q;
        float sum = 0.f;
#pragma unroll 8
        for (int j = 0; j < H; ++j) sum = fmaf(hid[(size_t)gi * H + j], Wh2[(size_t)j * Q + q], sum);
        lg[it] = sum;
        if (gi < ng) logits[(size_t)(g0 + gi) * Q + q] = sum;
    }
    __syncthreads();

    // ---- softmax + argmax over Q, a wavefront per graph
    if (probs || pred) {
        for (int gi = wave; gi < ng; gi += WAVES) {
            float* row = lg + (size_t)gi * Q;
            const int g = g0 + gi;
            const float first = row[0];
            float mx = first;                       // the reference scan starts at element 0
            float bv = -INFINITY;
            int bi = 0x7fffffff;
            for (int q = lane; q < Q; q += kWave) {
                const float v = row[q];
                mx = max_keep(mx, v);
                const float vv = (v != v) ? -INFINITY : v;     // a NaN that is not first never wins
                argmax_combine(bv, bi, vv, q);
            }
            mx = wave_max(mx);
            wave_argmax(bv, bi);
            if (first != first) bi = 0;             // a NaN in column 0 is never displaced
            if (pred && lane == 0) pred[g] = bi;
            if (probs) {
                float sum = 0.f;
                for (int q = lane; q < Q; q += kWave) {
                    const float e = expf(row[q] - mx);
                    row[q] = e;
                    sum += e;
                }
                sum = wave_sum(sum);
                for (int q = lane; q < Q; q += kWave) probs[(size_t)g * Q + q] = row[q] / sum;
            }
        }
    }
}

template <int C>
int launch_readout_tile(int B, int H, int Q, const int* s_row_ptr, const int* s_col_idx, const float* s_val,
                        const float* h, const float* Wh1, const float* Wh2, float* pool, float* hidden,
                        float* logits, float* probs, int* pred, hipStream_t s)
{
    const size_t smem = sizeof(float) * (size_t)kTileGraphs * ((size_t)C + 4 + H + Q);
    if (smem > 64 * 1024) return GNNHIP_EUNSUPPORTED;
    const unsigned grid = (unsigned)(((long long)B + kTileGraphs - 1) / kTileGraphs);
    // Sixteen wavefronts, a graph each, where the tiles are about one round of the two workgroups that a compute unit holds then, eight beyond
    // (hidden 256, 128 units, 30 nodes: 10,000 graphs 76.4 us with four, 71.8 with eight, 71.1 with sixteen, 4,097 33.7, 29.8 and 29.3; 12,288 of 25, 64
    // units 71.1, 67.4 and 72.4; hidden 128: 9,999 36.8, 34.4 and 32.9, 20,000 81.6, 79.7 and 85.9, 25,000 of 2 nodes 29.5, 29.0 and 33.4)
    const int waves = 2 * grid <= 5 * kNumCU ? 16 : 8;
    const auto kernel = waves == 16 ? &s2v_readout_tile_kernel<C, 16> : &s2v_readout_tile_kernel<C, 8>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(waves * kWave), smem, s, B, H, Q, s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2,
                       pool, hidden, logits, probs, pred);
    GNNHIP_LAUNCH_CHECK("s2v_readout_tile");
    return GNNHIP_OK;
}

// Readout for any hidden size up to 256 and any number of graphs: TG graphs per workgroup of BLOCK lanes, a quarter of it (one
// wavefront) or all of it per graph.
//   1. sum-pool   groups of G lanes (a power of two, 4 G >= C) take the graph's rows in turn, FLIGHT in flight each; the sums of a
//                 wavefront's groups are added by shuffles, those of the graph's wavefronts in order through LDS;
//   2. hidden     each wavefront of the graph adds up its share of the columns of W_h1, a lane per unit;
//   3. logits     a wavefront per class, lanes over the hidden units;
//   4. softmax and arg-max by the graph's first wavefront.
// Bound by memory where graphs are large (what is in flight decides: 301 graphs of 1,000 nodes, hidden 32: 17 us with two rows
// in flight per group of a 256-lane workgroup, 12 with eight of a 512-lane one, 18 with
// 1,024 lanes, which leave 45 of the workgroups to a second turn), by the chain of its four steps where they are
// small.  Hidden sizes without another readout took six launches (1,500 graphs of 32 nodes, hidden 100: 35 us).
//
// MINW: wavefronts per SIMD that the registers have to leave room for, 0: none asked for.  Only the variant with three rows in flight asks:
// where it does not change their number, asking only makes the compiler wait for each load by itself (a wavefront per graph, five
// asked for, which the kernel has anyway: 2,048 graphs of 24 nodes, hidden 160 16.1 -> 30.1 us, 256 21.6 -> 47.6).
template <int TG, int BLOCK, int MINW, int FLIGHT, bool POOL>
__global__ __launch_bounds__(BLOCK, MINW) void s2v_readout_rows_kernel(
    int B, int C, int H, int Q, const int* __restrict__ s_row_ptr, const int* __restrict__ s_col_idx, const float* __restrict__ s_val,
    const float* __restrict__ h, const float* __restrict__ Wh1, const float* __restrict__ Wh2, float* __restrict__ pool,
    float* __restrict__ hidden, float* __restrict__ logits, float* __restrict__ probs, int* __restrict__ pred, const int* __restrict__ gate)
{
    if (gated_off<POOL>(gate)) return;
    using V = ColsLoose;
    constexpr int LG = BLOCK / TG, WG = LG / kWave;      // lanes and wavefronts per graph
    constexpr int kFlight = FLIGHT;
    const int units = (C + 3) / 4, C4 = 4 * units;
    const int logG = units <= 1 ? 0 : 32 - __builtin_clz((unsigned)(units - 1));
    const int G = 1 << logG;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int k = tid / LG, w = (tid % LG) / kWave;      // graph of the tile, wavefront of the graph
    const int sub = lane & (G - 1), grp = (tid % LG) >> logG, ngroups = LG >> logG;
    const bool live = sub < units;
    const int col0 = V::at(sub, C);
    extern __shared__ float4 smem4[];
    float* part = reinterpret_cast<float*>(smem4) + (size_t)k * WG * C4;                     // [WG][C4], a unit's columns at 4 unit
    float* pl = reinterpret_cast<float*>(smem4) + (size_t)TG * WG * C4 + (size_t)k * C4;     // [C]
    float* ph = reinterpret_cast<float*>(smem4) + (size_t)TG * (WG + 1) * C4 + (size_t)k * (WG * H + H + Q);
    float* hid = ph + WG * H;                            // ph: [WG][H]
    float* lg = hid + H;

    for (long long tile = blockIdx.x; tile * TG < B; tile += gridDim.x) {
        const long long g = tile * TG + k;
        const bool own = g < B;
        const int start = own ? s_row_ptr[g] : 0, end = own ? s_row_ptr[g + 1] : 0;
        float4 acc = f4_zero();
        for (int t = start + grp; t < end; t += kFlight * ngroups) {
            int c[kFlight];
            float v[kFlight];
            float4 x[kFlight];
#pragma unroll
            for (int u = 0; u < kFlight; ++u) {
                const bool ok = t + u * ngroups < end;
                c[u] = ok ? s_col_idx[t + u * ngroups] : 0;
                v[u] = ok ? s_val[t + u * ngroups] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < kFlight; ++u) x[u] = live && t + u * ngroups < end ? V::load(h + (size_t)c[u] * C + col0) : f4_zero();
#pragma unroll
            for (int u = 0; u < kFlight; ++u)
                if (t + u * ngroups < end) f4_fma(acc, v[u], x[u]);
        }
        for (int d = G; d < kWave; d <<= 1)
            acc = V::add(acc, make_float4(__shfl_xor(acc.x, d, kWave), __shfl_xor(acc.y, d, kWave), __shfl_xor(acc.z, d, kWave), __shfl_xor(acc.w, d, kWave)));
        if (lane < units) *reinterpret_cast<float4*>(part + w * C4 + 4 * lane) = acc;
        __syncthreads();
        if (w == 0 && lane < units) {
            float4 s = *reinterpret_cast<const float4*>(part + 4 * lane);
#pragma unroll
            for (int i = 1; i < WG; ++i) s = V::add(s, *reinterpret_cast<const float4*>(part + i * C4 + 4 * lane));
            V::store(pl + V::at(lane, C), s);
            if (own) V::store(pool + (size_t)g * C + V::at(lane, C), s);
        }
        __syncthreads();
        if constexpr (POOL) continue;
        // ---- hidden = ReLU(pool * W_h1)
        const int share = (C + WG - 1) / WG, c_lo = min(w * share, C), c_hi = min(c_lo + share, C);
        for (int j = lane; j < H; j += kWave) {
            float s = 0.f;
#pragma unroll (2 * FLIGHT)
            for (int c = c_lo; c < c_hi; ++c) s = fmaf(pl[c], Wh1[(size_t)c * H + j], s);
            ph[w * H + j] = s;
        }
        __syncthreads();
        for (int j = tid % LG; j < H; j += LG) {
            float s = ph[j];
#pragma unroll
            for (int i = 1; i < WG; ++i) s += ph[i * H + j];
            s = relu_ref(s);
            hid[j] = s;
            if (own) hidden[(size_t)g * H + j] = s;
        }
        __syncthreads();
        // ---- logits = hidden * W_h2
        for (int q = w; q < Q; q += WG) {
            float s = 0.f;
            for (int j = lane; j < H; j += kWave) s = fmaf(hid[j], Wh2[(size_t)j * Q + q], s);
            s = wave_sum(s);
            if (lane == 0) {
                lg[q] = s;
                if (own) logits[(size_t)g * Q + q] = s;
            }
        }
        __syncthreads();
        // ---- softmax + argmax over Q
        if (w == 0 && own && (probs || pred)) {
            const float first = lg[0];
            float mx = first;                       // the reference scan starts at element 0
            float bv = -INFINITY;
            int bi = 0x7fffffff;
            for (int q = lane; q < Q; q += kWave) {
                const float v = lg[q];
                mx = max_keep(mx, v);
                argmax_combine(bv, bi, (v != v) ? -INFINITY : v, q);     // a NaN that is not first never wins
            }
            mx = wave_max(mx);
            wave_argmax(bv, bi);
            if (first != first) bi = 0;             // a NaN in column 0 is never displaced
            if (pred && lane == 0) pred[g] = bi;
            if (probs) {
                float s = 0.f;
                for (int q = lane; q < Q; q += kWave) {
                    const float e = expf(lg[q] - mx);
                    lg[q] = e;
                    s += e;
                }
                s = wave_sum(s);
                for (int q = lane; q < Q; q += kWave) probs[(size_t)g * Q + q] = lg[q] / s;
            }
        }
        __syncthreads();                            // LDS is reused by the next tile
    }
}

template <int TG, int BLOCK, int MINW, int FLIGHT, bool POOL = false>
int launch_readout_rows(int B, int C, int H, int Q, const int* s_row_ptr, const int* s_col_idx, const float* s_val, const float* h,
                        const float* Wh1, const float* Wh2, float* pool, float* hidden, float* logits, float* probs, int* pred, hipStream_t s,
                        const int* gate = nullptr)
{
    constexpr int WG = BLOCK / TG / kWave;
    const size_t smem = sizeof(float) * TG * ((size_t)(WG + 1) * ((C + 3) / 4 * 4) + (size_t)(WG + 1) * H + Q);
    if (smem > 64 * 1024) return GNNHIP_EUNSUPPORTED;
    const int tiles = (B + TG - 1) / TG, most = kNumCU * (2048 / BLOCK);
    hipLaunchKernelGGL((s2v_readout_rows_kernel<TG, BLOCK, MINW, FLIGHT, POOL>), dim3((unsigned)(tiles < most ? tiles : most)), dim3(BLOCK), smem, s, B, C, H, Q,
                       s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2, pool, hidden, logits, probs, pred, gate);
    GNNHIP_LAUNCH_CHECK("s2v_readout_rows");
    return GNNHIP_OK;
}

// over 16 lanes
__device__ __forceinline__ float row_sum(float v)
{
    v += dpp_mov_f<kDppXor1>(v);
    v += dpp_mov_f<kDppXor2>(v);
    v += dpp_mov_f<kDppHalfMirror>(v);
    return v + dpp_mov_f<kDppMirror>(v);
}

__device__ __forceinline__ float row_max(float v)
{
    v = max_keep(v, dpp_mov_f<kDppXor1>(v));
    v = max_keep(v, dpp_mov_f<kDppXor2>(v));
    v = max_keep(v, dpp_mov_f<kDppHalfMirror>(v));
    return max_keep(v, dpp_mov_f<kDppMirror>(v));
}

__device__ __forceinline__ void row_argmax(float& v, int& i)
{
    argmax_combine(v, i, dpp_mov_f<kDppXor1>(v), dpp_mov_i<kDppXor1>(i));
    argmax_combine(v, i, dpp_mov_f<kDppXor2>(v), dpp_mov_i<kDppXor2>(i));
    argmax_combine(v, i, dpp_mov_f<kDppHalfMirror>(v), dpp_mov_i<kDppHalfMirror>(i));
    argmax_combine(v, i, dpp_mov_f<kDppMirror>(v), dpp_mov_i<kDppMirror>(i));
}

// The readout behind pooled rows that are there, a workgroup per 16 graphs: a wavefront forms the hidden layer in blocks of 16 units on the FP32 matrix
// cores, both operands straight from memory, up to 64 columns in one trip; then 16 lanes per graph add up its logits, a unit in 16 each, and
// do softmax and arg-max.  Bound by the chain of its steps.  30,000 graphs, hidden 64, 32 units:
// 13 us in a trace; the wavefront-per-graph kernel from its second step on 33, a lane per unit and four graphs with LDS operands 17.
constexpr int kPooledGraphs = 16;
constexpr int kPooledWaves = 4;

__global__ __launch_bounds__(kPooledWaves * kWave) void s2v_readout_pooled_kernel(int B, int C, int H, int Q, const float* __restrict__ pool,
                                                                                  const float* __restrict__ Wh1, const float* __restrict__ Wh2,
                                                                                  float* __restrict__ hidden, float* __restrict__ logits,
                                                                                  float* __restrict__ probs, int* __restrict__ pred)
{
    constexpr int kSteps = 16;                       // contraction steps of a trip, four columns each
    extern __shared__ float smem[];
    const int ldh = H | 1;
    float* hid = smem;                               // [kPooledGraphs][ldh]
    float* lg = hid + (size_t)kPooledGraphs * ldh;   // [kPooledGraphs][Q]
    float* w2 = lg + (size_t)kPooledGraphs * Q;      // [H][Q]
    constexpr int kThreads = kPooledWaves * kWave;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), q = lane >> 4, t = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int g0 = (int)blockIdx.x * kPooledGraphs, ng = min(kPooledGraphs, B - g0);
    const float w2_first = Wh2[min(tid, H * Q - 1)];

    // ---- hidden = ReLU(pool * W_h1), transposed: lane (q, t) ends up with units 4 q .. of graph t
    const float* row = pool + (size_t)(g0 + min(t, ng - 1)) * C;
    for (int j0 = 16 * wave; j0 < H; j0 += 16 * kPooledWaves) {
        const float* col = Wh1 + min(j0 + t, H - 1);
        mfma_f4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int c0 = 0; c0 < C; c0 += 4 * kSteps) {
            float x[kSteps], w[kSteps];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const int c = min(c0 + 4 * s + q, C - 1);
                x[s] = row[c];
                w[s] = col[c * H];
            }
            __builtin_amdgcn_sched_barrier(0);       // all of them in flight
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const bool in = c0 + 4 * s + q < C;  // both are zero past the last column
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? w[s] : 0.f, in ? x[s] : 0.f, acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = j0 + 4 * q + i;
            const float v = relu_ref(acc[i]);
            if (j < H) {
                hid[t * ldh + j] = v;
                if (t < ng) hidden[(size_t)(g0 + t) * H + j] = v;
            }
        }
    }
    if (tid < H * Q) w2[tid] = w2_first;
    for (int i = tid + kThreads; i < H * Q; i += kThreads) w2[i] = Wh2[i];
    __syncthreads();

    // ---- logits = hidden * W_h2, softmax + argmax over Q
    static_assert(kThreads == 16 * kPooledGraphs, "16 lanes per graph");
    const int g = tid / 16, sub = t;
    float* logit = lg + (size_t)g * Q;
    for (int c = 0; c < Q; ++c) {
        float s = 0.f;
        for (int j = sub; j < H; j += 16) s = fmaf(hid[g * ldh + j], w2[j * Q + c], s);
        s = row_sum(s);
        if (sub == 0) logit[c] = s;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const float first = logit[0];
    float mx = first;                                // the reference scan starts at element 0
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for (int c = sub; c < Q; c += 16) {
        const float v = logit[c];
        if (g < ng) logits[(size_t)(g0 + g) * Q + c] = v;
        mx = max_keep(mx, v);
        argmax_combine(bv, bi, (v != v) ? -INFINITY : v, c);          // a NaN that is not first never wins
    }
    if (pred) {
        row_argmax(bv, bi);
        if (first != first) bi = 0;                  // a NaN in column 0 is never displaced
        if (sub == 0 && g < ng) pred[g0 + g] = bi;
    }
    if (probs) {
        mx = row_max(mx);
        float s = 0.f;
        for (int c = sub; c < Q; c += 16) {
            const float e = expf(logit[c] - mx);
            logit[c] = e;
            s += e;
        }
        s = row_sum(s);
        if (g < ng)
            for (int c = sub; c < Q; c += 16) probs[(size_t)(g0 + g) * Q + c] = logit[c] / s;
    }
}

}  // namespace

// A workgroup per tile of graphs, hidden sizes 128 and 256; for batches of thousands of small graphs (the caller decides).
int readout_tile_dispatch(int B, int C, int H, int Q, const int* s_row_ptr, const int* s_col_idx, const float* s_val,
                          const float* h, const float* Wh1, const float* Wh2, float* pool, float* hidden,
                          float* logits, float* probs, int* pred, hipStream_t s)
{
    if (!aligned16(h) || !aligned16(pool) || B <= 0) return GNNHIP_EUNSUPPORTED;
#define GNNHIP_RO_ARGS B, H, Q, s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2, pool, hidden, logits, probs, pred, s
    switch (C) {
    case 128: return launch_readout_tile<128>(GNNHIP_RO_ARGS);
    case 256: return launch_readout_tile<256>(GNNHIP_RO_ARGS);
    }
#undef GNNHIP_RO_ARGS
    return GNNHIP_EUNSUPPORTED;
}

// One wavefront per graph; for batches of many graphs (the caller decides).  Returns GNNHIP_EUNSUPPORTED
// for hidden sizes it has no kernel for and when W_h1 and W_h2 do not fit LDS.
int readout_wave_dispatch(int B, int C, int H, int Q, const int* s_row_ptr, const int* s_col_idx, const float* s_val,
                          const float* h, const float* Wh1, const float* Wh2, float* pool, float* hidden,
                          float* logits, float* probs, int* pred, hipStream_t s)
{
    if (!aligned16(h)) return GNNHIP_EUNSUPPORTED;
#define GNNHIP_RO_ARGS B, H, Q, s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2, pool, hidden, logits, probs, pred, s
    switch (C) {
    case 16: return launch_readout_wave<16>(GNNHIP_RO_ARGS);
    case 32: return launch_readout_wave<32>(GNNHIP_RO_ARGS);
    case 64: return launch_readout_wave<64>(GNNHIP_RO_ARGS);
    }
#undef GNNHIP_RO_ARGS
    return GNNHIP_EUNSUPPORTED;
}

// Any hidden size of 4 .. 256.
int readout_rows_dispatch(int B, int N, int C, int H, int Q, const int* s_row_ptr, const int* s_col_idx, const float* s_val, const float* h,
                          const float* Wh1, const float* Wh2, float* pool, float* hidden, float* logits, float* probs, int* pred, hipStream_t s)
{
    if (C < 4 || C > 256) return GNNHIP_EUNSUPPORTED;
#define GNNHIP_RO_ARGS B, C, H, Q, s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2, pool, hidden, logits, probs, pred, s
    // Many small graphs: a wavefront each (4,000 graphs of 32 nodes, hidden 100: 22 us, with a workgroup each 29; 1,500 of them:
    // 16.6 against 15.6).  Graphs of hundreds of rows: 512 lanes each.
    const long long mean = (long long)N / B;
    int rc = GNNHIP_EUNSUPPORTED;
    // 1,025 to 1,536 small graphs, a workgroup each: three rows in flight per group take 74 registers, which leaves six workgroups per
    // compute unit where eight take 108 and leave four and a second wave of workgroups (24 nodes each, 1,500 graphs: hidden 48
    // 11.4 -> 6.6 us, 100 11.6 -> 7.7, 200 14.6 -> 11.3; 250 nodes each: hidden 48 23.1 -> 18.2, 33 20.5 -> 16.5 and, at 1,025 graphs,
    // 14.6 -> 14.9).  Past 1,536 there are two waves either way, and hidden 200 loses 8 %; below 1,025 there is one, and which is
    // faster changes with the width (hidden 48, 600 graphs of 60: 6.7 -> 5.9; 64: 6.1 -> 6.3; 200: 11.6 -> 15).
    int lanes = 1;
    while (4 * lanes < C) lanes *= 2;
    const long long turn = mean * lanes;                 // lanes that the rows of a graph take together
    const bool few = B > 4 * kNumCU && B <= 6 * kNumCU && turn <= 16 * kBlock;
    if (B >= 8 * kNumCU && mean <= 256) rc = launch_readout_rows<4, kBlock, 0, 8>(GNNHIP_RO_ARGS);
    else if (mean > 256) rc = launch_readout_rows<1, 512, 0, 8>(GNNHIP_RO_ARGS);
    if (rc == GNNHIP_EUNSUPPORTED && few) rc = launch_readout_rows<1, kBlock, 6, 3>(GNNHIP_RO_ARGS);
    if (rc == GNNHIP_EUNSUPPORTED) rc = launch_readout_rows<1, kBlock, 0, 8>(GNNHIP_RO_ARGS);
    return rc;
#undef GNNHIP_RO_ARGS
}

size_t pooled_lds_bytes(int H, int Q) { return sizeof(float) * ((size_t)kPooledGraphs * ((H | 1) + Q) + (size_t)H * Q); }

// whether readout_gated_dispatch takes these sizes; that its first launch does follows (four of its wavefronts take 5 C and 5 H words)
bool readout_gated_accepts(int C, int H, int Q) { return C >= 4 && C <= 256 && pooled_lds_bytes(H, Q) <= 64 * 1024; }

// The readout behind the one launch of a batch's levels, which has added up the pooled rows: those again if the gate says so, and what follows
// them.  Eight rows in flight per group at any size: three, which the whole readout takes for 1,025 to 1,536 graphs, are slower for the pooled rows
// alone (1,200 graphs of 90 nodes, hidden 50, a forward of four levels 146.8 us, 149.7 with three).
int readout_gated_dispatch(int B, int C, int H, int Q, bool wave, const int* s_row_ptr, const int* s_col_idx, const float* s_val, const float* h,
                           const float* Wh1, const float* Wh2, float* pool, float* hidden, float* logits, float* probs, int* pred,
                           hipStream_t s, const int* gate)
{
#define GNNHIP_RO_ARGS H, Q, s_row_ptr, s_col_idx, s_val, h, Wh1, Wh2, pool, hidden, logits, probs, pred, s, gate
    int rc = GNNHIP_EUNSUPPORTED;
    if (wave && aligned16(h)) {
        switch (C) {                                     // (hidden 16 has no pooled rows: batch_levels_with_pool)
        case 32: rc = launch_readout_wave<32, true>(B, GNNHIP_RO_ARGS); break;
        case 64: rc = launch_readout_wave<64, true>(B, GNNHIP_RO_ARGS); break;
        }
    }
    if (rc == GNNHIP_EUNSUPPORTED && B >= 8 * kNumCU) rc = launch_readout_rows<4, kBlock, 0, 8, true>(B, C, GNNHIP_RO_ARGS);
    if (rc == GNNHIP_EUNSUPPORTED) rc = launch_readout_rows<1, kBlock, 0, 8, true>(B, C, GNNHIP_RO_ARGS);
#undef GNNHIP_RO_ARGS
    if (rc) return rc;
    hipLaunchKernelGGL(s2v_readout_pooled_kernel, dim3(ceil_div_u((size_t)B, kPooledGraphs)), dim3(kPooledWaves * kWave), pooled_lds_bytes(H, Q), s, B, C, H, Q, pool, Wh1, Wh2,
                       hidden, logits, probs, pred);
    GNNHIP_LAUNCH_CHECK("s2v_readout_pooled");
    return GNNHIP_OK;
}

}  // namespace gnnhip
