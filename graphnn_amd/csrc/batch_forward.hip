// Input stage and all levels of the inference forward in one launch, for batches that turn out to be many small graphs.
//
//     msg = X W_n2l ;  h_0 = ReLU(msg) ;  L times  h <- ReLU((A h) W + msg)
//     (examples/graph_classification/src/kernel_mean_field.cpp:31-44)
//
// The general forward knows nothing about its batch, so this kernel finds out on the device whether it may run: the ranges of
// nodes that the rows of S stand for are cut into bins of up to kRows nodes (graph_bins.h), a workgroup takes a bin, and an entry of A
// that leaves its bin, or rows of S that are no such ranges, set *refused.  The launches of the level-by-level route follow
// behind it and do nothing unless that word is set, so a batch of any other kind comes out as it always did.
//
// Level by level such a batch is bound by memory: every level reads h and msg and writes h, 3.3 GB for 880,690 nodes at hidden 64.
// Here the rows of a bin stay in LDS and msg in registers: X and the entries are read once, msg and the last h written once
// (0.6 GB).  880,690 nodes, four levels, the whole forward: hidden 64 768 -> 443 us, hidden 32 419 -> 230; a level more 158 -> 55 and
// 87 -> 30.
//
// A wavefront owns 16 or 32 rows and all their columns.  Lane (q = lane / 16, t = lane % 16) holds columns KS q .. KS q + KS - 1 of
// row t, in every role: it sums that part of the row's neighbours straight into the operand registers of the matrix
// instructions (contraction step s takes k = KS q + s), it ends up with that part of the product (the columns of W are taken in
// that order), and adds that part of msg.  Nothing is passed between lanes, and a level has two barriers: h is
// rewritten in place when every row has been summed.
//
// Hidden 16 and 32 run on the FP32 matrix cores; the order of the sums is that of level_stream.hip and graph_forward.hip, so
// every bit of h is theirs.  At hidden 64 the FP32 matrix instructions were the longest part (480 us of a kernel that takes 380
// now), so its products are formed from bf16 pieces (bf16_split.h), the first two pieces of W in registers: rms error against float64
// 1.16e-11 of the terms' magnitudes after four levels, level by level 2.42e-11.  What bounds that kernel is the issue of vector
// instructions, about 330 per 16 rows and level (64 sum the first four entries, 104 split the rows); two wavefronts per SIMD, 247
// registers.  What a bin reads is asked for while the last level of the bin before it ends (428 us without).
#include <type_traits>

#include "bf16_split.h"
#include "columns.h"
#include "graph_bins.h"

namespace gnnhip {
namespace {

constexpr int kRows = 128;                       // nodes of a bin
constexpr int kEdgeCap = 1024;                   // entries of a bin kept in LDS; those of a bin with more are read from memory in every level
constexpr int kDirect = 4;                       // entries per row whose place and weight stay in registers

// ReLU as one instruction: NaN passes, as in relu_ref4, but -0 becomes 0 (two instructions cost 3 % of a level in pieces, where nothing
// else is the same to the bit either)
__device__ __forceinline__ float4 relu_one(const float4& v)
{
    return make_float4(__builtin_elementwise_maximum(v.x, 0.f), __builtin_elementwise_maximum(v.y, 0.f), __builtin_elementwise_maximum(v.z, 0.f),
                       __builtin_elementwise_maximum(v.w, 0.f));
}

template <int C> struct BatchShape;
// TPW: tiles of 16 rows per wavefront.  MINW: wavefronts per SIMD.  PIECES: products from bf16 pieces
template <> struct BatchShape<16> { static constexpr int TPW = 1, MINW = 6; static constexpr bool PIECES = false; };
template <> struct BatchShape<32> { static constexpr int TPW = 1, MINW = 4; static constexpr bool PIECES = false; };
template <> struct BatchShape<64> { static constexpr int TPW = 2, MINW = 2; static constexpr bool PIECES = true; };
template <int C> constexpr int batch_waves() { return kRows / 16 / BatchShape<C>::TPW; }

template <int C, int KSX>
constexpr size_t batch_lds_bytes()
{
    return sizeof(float) * (size_t)(kRows + 1) * (C + 4) + (BatchShape<C>::PIECES ? sizeof(float) * C + sizeof(short) * C * C : 0) +
           sizeof(float) * (size_t)(C / 16) * KSX * kWave + sizeof(int2) * kEdgeCap + sizeof(int) * (kRows + 4);
}

// KSX: contraction steps of the input stage, K <= 4 KSX
template <int C, int KSX>
__global__ __launch_bounds__(batch_waves<C>() * kWave, BatchShape<C>::MINW) void s2v_batch_levels_kernel(
    int N, int B, int K, int L, const int* __restrict__ a_row_ptr, const int* __restrict__ a_col_idx, const float* __restrict__ a_val,
    const float* __restrict__ X, const float* __restrict__ Wn2l, const float* __restrict__ Wc, float* __restrict__ msg,
    float* __restrict__ h_out, const int* __restrict__ bins, int* __restrict__ refused)
{
    constexpr int TPW = BatchShape<C>::TPW, kWaves = batch_waves<C>(), kBlock = kWaves * kWave;
    constexpr bool PIECES = BatchShape<C>::PIECES;
    constexpr int KS = C / 4;                    // columns of a lane, contraction steps of a level
    constexpr int KS2 = C / 32;                  // contraction steps of a level in pieces
    constexpr int NJB = C / 16;                  // output blocks of 16 columns
    constexpr int LD = C + 4;
    static_assert(!PIECES || KS2 == 2, "two sums of opposite signs");
    extern __shared__ float4 smem4[];
    float* hbuf = reinterpret_cast<float*>(smem4);                         // [kRows + 1][LD], the last row zeros
    bf16_words4* w3 = reinterpret_cast<bf16_words4*>(hbuf + (kRows + 1) * LD);             // third pieces of W, [KS2][NJB][lane]
    float* w_down = reinterpret_cast<float*>(w3 + (PIECES ? KS2 * NJB * kWave : 0));       // [C] a column's scale up over its scale
    float2* wn = reinterpret_cast<float2*>(w_down + (PIECES ? C : 0));     // [NJB][KSX / 2][lane]
    int2* edges = reinterpret_cast<int2*>(wn + NJB * (KSX / 2) * kWave);   // [kEdgeCap] row offset, weight
    int* rp = reinterpret_cast<int*>(edges + kEdgeCap);                    // [kRows + 1], from the bin's first entry on
    __shared__ int stop;                         // another workgroup has come upon an entry that leaves its bin
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int row0 = 16 * TPW * wave + t;        // this lane's row of the bin in the wavefront's first tile
    const int out_col = KS * (t >> 2) + (t & 3); // column of W that a lane supplies to block jb: out_col + 4 jb
    // contraction steps of the input stage that are needed.  Steps 2 j and 2 j + 1 take k = 8 j + 2 q and the one behind it, so that a load of
    // a pair of columns by all lanes covers 32 consecutive bytes of 16 rows
    const int srt = 2 * ((K + 7) / 8);

    BinFinder finder(B, bins);
    int at = finder.find_checked((int)blockIdx.x);

    // W as the operand of the matrix instructions.  fp32: wf[jb][s] = W[KS q + s][out_col + 4 jb]; in pieces: of W[KS q + 8 s + 0..7],
    // the third ones in LDS, the second step's negated
    float wf[PIECES ? 1 : NJB][PIECES ? 1 : KS];
    bf16_words4 wp[PIECES ? KS2 : 1][PIECES ? NJB : 1][2];
    bool any_down = false;                       // a column of W is scaled down (bf16_split.h): uniform
    if constexpr (PIECES) {
#pragma unroll
        for (int jb = 0; jb < NJB; ++jb) {
            float w[KS], largest = 0.f;
#pragma unroll
            for (int k = 0; k < KS; ++k) w[k] = Wc[(size_t)(KS * q + k) * C + out_col + 4 * jb];
#pragma unroll
            for (int k = 0; k < KS; k += 2) largest = split_max(largest, w[k], w[k + 1]);
            const unsigned long long large = __ballot(largest >= kSplitLarge);
            const bool down = (large >> t) & 0x0001000100010001ull;        // in any quarter of the column
            any_down |= large != 0;
            const float scale = down ? kSplitDown : kSplitUp;
            if (q == 0) w_down[out_col + 4 * jb] = down ? kSplitUp / kSplitDown : 1.f;
#pragma unroll
            for (int s = 0; s < KS2; ++s) {
                bf16_words4 third;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    unsigned p[3];
                    bf16_split2(w[8 * s + 2 * i] * scale, w[8 * s + 2 * i + 1] * scale, down, p);
                    const unsigned sign = s == 1 ? 0x80008000u : 0u;
                    wp[s][jb][0][i] = p[0] ^ sign; wp[s][jb][1][i] = p[1] ^ sign; third[i] = p[2] ^ sign;
                }
                if (wave == 0) w3[(s * NJB + jb) * kWave + lane] = third;
            }
        }
    } else {
#pragma unroll
        for (int jb = 0; jb < NJB; ++jb)
#pragma unroll
            for (int s = 0; s < KS; ++s) wf[jb][s] = Wc[(size_t)(KS * q + s) * C + out_col + 4 * jb];
    }
    for (int i = wave; i < NJB * (KSX / 2); i += kWaves) {
        const int jb = i / (KSX / 2), k = 8 * (i % (KSX / 2)) + 2 * q;
        wn[i * kWave + lane] = make_float2(k < K ? Wn2l[(size_t)k * C + out_col + 4 * jb] : 0.f,
                                           k + 1 < K ? Wn2l[(size_t)(k + 1) * C + out_col + 4 * jb] : 0.f);
    }
    if (tid < LD) hbuf[kRows * LD + tid] = 0.f;
    if (tid == 0) stop = 0;
    __syncthreads();

    // ---- what a bin needs from memory, asked for together and a bin ahead
    struct Bin { int node0, n, e0, ne; };
    auto record = [&](int at) {
        const int* rec = bins + bin_words_ints(B) + (size_t)max(at, 0) * kOrderRec;
        const int4 r = *reinterpret_cast<const int4*>(rec);
        return at < 0 ? Bin{0, 0, 0, 0} : Bin{r.y, r.z, r.w, max(rec[4] - r.w, 0)};
    };
    constexpr int kEdgesEach = kEdgeCap / kBlock;
    float x[TPW][KSX], e_val[kEdgesEach];
    int e_col[kEdgesEach], rp_v;
    auto ask = [&](const Bin& b) {
        // (every register is written whatever the bin is, or the old values would have to be kept through the levels)
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            const float* xr = X + (size_t)min(b.node0 + min(row0 + 16 * i, max(b.n - 1, 0)), N - 1) * K;
#pragma unroll
            for (int s = 0; s < KSX; s += 2) {
                if (s >= srt) { x[i][s] = x[i][s + 1] = 0.f; continue; }        // uniform
                // a pair of columns per load (K >= 2); the last one may repeat a column
                typedef float f32x2_at4 __attribute__((ext_vector_type(2), aligned(4)));
                const f32x2_at4 v = *reinterpret_cast<const f32x2_at4*>(xr + min(4 * s + 2 * q, K - 2));
                x[i][s] = v.x; x[i][s + 1] = v.y;
            }
        }
        rp_v = a_row_ptr[b.node0 + min(tid, b.n)];
        const int in_lds = b.ne <= kEdgeCap ? b.ne : 0;
#pragma unroll
        for (int u = 0; u < kEdgesEach; ++u) {
            const int e = tid + u * kBlock;
            e_col[u] = e < in_lds ? a_col_idx[b.e0 + e] : 0;
            e_val[u] = e < in_lds ? a_val[b.e0 + e] : 0.f;
        }
    };
    Bin cur = record(at), next;
    bool more = at >= 0;                         // there is a bin `cur`
    ask(cur);

    for (int bin = blockIdx.x; more && !stop; bin += gridDim.x) {
        // (the same in all wavefronts: stop is written between two barriers that this test does not lie between)
        const int node0 = cur.node0, n = cur.n, e0 = cur.e0, ne = cur.ne;
        const bool staged = ne <= kEdgeCap;
        const int tiles = min(max((n + 15) / 16 - TPW * wave, 0), TPW);    // of this wavefront: uniform
        if (tid <= n) rp[tid] = rp_v - e0;
        if (staged) {
#pragma unroll
            for (int u = 0; u < kEdgesEach; ++u) {
                const int e = tid + u * kBlock;
                if (e < ne) {
                    const int c = e_col[u] - node0;
                    if (c < 0 || c >= n) *refused = 1;
                    edges[e] = make_int2(min(max(c, 0), n - 1) * LD, __float_as_int(e_val[u]));
                }
            }
        }
        at = finder.find_checked(bin + (int)gridDim.x);
        more = at >= 0;
        next = record(at);

        // ---- input stage
        float4 m[TPW][NJB];
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            mfma_f4 acc[NJB];
#pragma unroll
            for (int jb = 0; jb < NJB; ++jb) acc[jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};
            if (i < tiles) {
#pragma unroll
                for (int s = 0; s < KSX; s += 2) {
                    if (s >= srt) continue;
                    const int past = 4 * s + 2 * q - (K - 2);         // the pair (k, k + 1); past > 0: the loads gave the last two columns
                    x[i][s] = past <= 0 ? x[i][s] : past == 1 ? x[i][s + 1] : 0.f;
                    x[i][s + 1] = past <= 0 ? x[i][s + 1] : 0.f;
#pragma unroll
                    for (int jb = 0; jb < NJB; ++jb) {
                        const float2 w = wn[(jb * (KSX / 2) + s / 2) * kWave + lane];
                        acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, x[i][s], acc[jb], 0, 0, 0);
                        acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, x[i][s + 1], acc[jb], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int jb = 0; jb < NJB; ++jb)
                m[i][jb] = row0 + 16 * i < n ? make_float4(acc[jb][0], acc[jb][1], acc[jb][2], acc[jb][3]) : f4_zero();
        }
        __syncthreads();                         // the last bin's rows have left hbuf; rp and edges are there
        float* own = hbuf + row0 * LD + KS * q;
        int g_st[TPW], g_en[TPW], g_off[TPW][kDirect];
        float g_w[TPW][kDirect];
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
#pragma unroll
            for (int jb = 0; jb < NJB; ++jb) *reinterpret_cast<float4*>(own + 16 * i * LD + 4 * jb) = m[i][jb];
            const int row = row0 + 16 * i;
            g_st[i] = g_en[i] = 0;
            if (row < n) { g_st[i] = rp[row]; g_en[i] = rp[row + 1]; }
#pragma unroll
            for (int u = 0; u < kDirect; ++u) {
                const bool ok = staged && g_st[i] + u < g_en[i];           // a missing entry is weight 0 times the row of zeros
                const int2 ed = edges[ok ? g_st[i] + u : 0];
                g_off[i][u] = (ok ? ed.x : kRows * LD) + KS * q;
                g_w[i][u] = ok ? __int_as_float(ed.y) : 0.f;
            }
        }
        __syncthreads();
        // the bin's rows as they lie in memory: whole lines
        auto copy_out = [&](float* dst) {
            for (int i = tid; i < n * KS; i += kBlock)
                *reinterpret_cast<float4*>(dst + (size_t)node0 * C + 4 * i) = *reinterpret_cast<const float4*>(hbuf + (i / KS) * LD + 4 * (i % KS));
        };
        copy_out(msg);
        if (tid == 0) stop = __hip_atomic_load(refused, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

        auto level = [&](auto relu_in, auto last) {
            constexpr bool kRelu = decltype(relu_in)::value;
            float4 v[TPW][NJB];
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                if (i >= tiles) continue;        // uniform
                float agg[KS];
#pragma unroll
                for (int k = 0; k < KS; ++k) agg[k] = 0.f;
                auto add = [&](int off, float w) {
#pragma unroll
                    for (int k = 0; k < KS; k += 4) {
                        float4 r = *reinterpret_cast<const float4*>(hbuf + off + k);
                        if (kRelu) r = PIECES ? relu_one(r) : relu_ref4(r);
                        agg[k] += w * r.x; agg[k + 1] += w * r.y; agg[k + 2] += w * r.z; agg[k + 3] += w * r.w;
                    }
                };
                if (staged) {
#pragma unroll
                    for (int u = 0; u < kDirect; ++u) add(g_off[i][u], g_w[i][u]);
                    for (int e = g_st[i] + kDirect; e < g_en[i]; ++e) {
                        const int2 ed = edges[e];
                        add(ed.x + KS * q, __int_as_float(ed.y));
                    }
                } else {
                    for (int e = g_st[i]; e < g_en[i]; ++e) {
                        const int c = a_col_idx[e0 + e] - node0;
                        if (c < 0 || c >= n) *refused = 1;
                        add(min(max(c, 0), n - 1) * LD + KS * q, a_val[e0 + e]);
                    }
                }
                if constexpr (PIECES) {
                    // the row in pieces, scaled (bf16_split.h)
                    bf16_words4 p[KS2][3];
                    float largest = 0.f, back = kSplitUpBack * kSplitUpBack;
#pragma unroll
                    for (int k = 0; k < KS; k += 2) largest = split_max(largest, agg[k], agg[k + 1]);
                    const unsigned long long large = __ballot(largest >= kSplitLarge);
                    auto split = [&](float scale, bool down) {
#pragma unroll
                        for (int s = 0; s < KS2; ++s)
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                unsigned w[3];
                                bf16_split2(agg[8 * s + 2 * u] * scale, agg[8 * s + 2 * u + 1] * scale, down, w);
                                p[s][0][u] = w[0]; p[s][1][u] = w[1]; p[s][2][u] = w[2];
                            }
                    };
                    if (large) {                 // uniform: some row is scaled down
                        const bool down = (large >> t) & 0x0001000100010001ull;
                        split(down ? kSplitDown : kSplitUp, down);
                        if (down) back = kSplitDownBack * kSplitUpBack;
                    } else {
                        split(kSplitUp, false);
                    }
                    // the corrections of either step first; the second step on a sum of the other sign, so that the drifts cancel
                    mfma_f4 acc[KS2][NJB];
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_bf16(w3[(s * NJB + jb) * kWave + lane], p[s][0], acc[s][jb]);
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_bf16(wp[s][jb][0], p[s][2], acc[s][jb]);
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_bf16(wp[s][jb][1], p[s][1], acc[s][jb]);
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_bf16(wp[s][jb][1], p[s][0], acc[s][jb]);
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_bf16(wp[s][jb][0], p[s][1], acc[s][jb]);
#pragma unroll
                    for (int s = 0; s < KS2; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[s][jb] = mfma_bf16(wp[s][jb][0], p[s][0], acc[s][jb]);
#pragma unroll
                    for (int jb = 0; jb < NJB; ++jb) {
                        float4 f = make_float4(back, back, back, back);
                        if (any_down) {
                            const float4 d = *reinterpret_cast<const float4*>(w_down + KS * q + 4 * jb);
                            f.x *= d.x; f.y *= d.y; f.z *= d.z; f.w *= d.w;
                        }
                        const mfma_f4 r = acc[0][jb] - acc[1][jb];
                        v[i][jb] = relu_one(make_float4(fmaf(r[0], f.x, m[i][jb].x), fmaf(r[1], f.y, m[i][jb].y), fmaf(r[2], f.z, m[i][jb].z),
                                                         fmaf(r[3], f.w, m[i][jb].w)));
                    }
                } else {
                    mfma_f4 acc[NJB];
#pragma unroll
                    for (int jb = 0; jb < NJB; ++jb) acc[jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < KS; ++s)
#pragma unroll
                        for (int jb = 0; jb < NJB; ++jb) acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[jb][s], agg[s], acc[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NJB; ++jb)
                        v[i][jb] = relu_ref4(make_float4(acc[jb][0] + m[i][jb].x, acc[jb][1] + m[i][jb].y, acc[jb][2] + m[i][jb].z, acc[jb][3] + m[i][jb].w));
                }
            }
            if constexpr (decltype(last)::value) ask(next);      // ahead of this bin's stores
            __syncthreads();                     // every row of the old embedding has been read
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                if (i >= tiles) continue;
#pragma unroll
                for (int jb = 0; jb < NJB; ++jb) *reinterpret_cast<float4*>(own + 16 * i * LD + 4 * jb) = v[i][jb];
            }
            __syncthreads();
        };
        if (L == 1) {
            level(std::true_type(), std::true_type());
        } else {
            level(std::true_type(), std::false_type());
            for (int lv = 2; lv < L; ++lv) level(std::false_type(), std::false_type());
            level(std::false_type(), std::true_type());
        }
        copy_out(h_out);
        cur = next;
    }
    // a segment that was not packed: every workgroup comes by all words
    if (finder.unpacked && tid == 0) *refused = 1;
}

template <int C, int KSX>
int launch_batch_levels(int N, int B, int K, int L, const int* a_row_ptr, const int* a_col_idx, const float* a_val, const float* X,
                        const float* Wn2l, const float* Wc, float* msg, float* h_out, const int* bins, int* refused, hipStream_t s)
{
    constexpr size_t smem = batch_lds_bytes<C, KSX>();
    static LdsLimit lds_limit;
    GNNHIP_HIP(lds_limit.raise(reinterpret_cast<const void*>(&s2v_batch_levels_kernel<C, KSX>), smem));
    // two neighbouring bins hold more than kRows nodes together, and every 64 graphs may leave one bin short
    long long most = 2ll * N / kRows + (B + kWave - 1) / kWave + 1;
    if (most > B) most = B;
    constexpr int kWaves = batch_waves<C>();
    const long long resident = (long long)kNumCU * (BatchShape<C>::MINW * 4 / kWaves);
    const unsigned grid = (unsigned)(most < resident ? most : resident);
    hipLaunchKernelGGL((s2v_batch_levels_kernel<C, KSX>), dim3(grid), dim3(kWaves * kWave), smem, s, N, B, K, L, a_row_ptr, a_col_idx, a_val, X, Wn2l,
                       Wc, msg, h_out, bins, refused);
    GNNHIP_LAUNCH_CHECK("s2v_batch_levels");
    return GNNHIP_OK;
}

template <int C>
int batch_levels_c(int N, int B, int K, int L, const int* a_row_ptr, const int* a_col_idx, const float* a_val, const float* X,
                   const float* Wn2l, const float* Wc, float* msg, float* h_out, const int* bins, int* refused, hipStream_t s)
{
#define GNNHIP_BL_ARGS N, B, K, L, a_row_ptr, a_col_idx, a_val, X, Wn2l, Wc, msg, h_out, bins, refused, s
    if (K <= 16) return launch_batch_levels<C, 4>(GNNHIP_BL_ARGS);
    if (K <= 32) return launch_batch_levels<C, 8>(GNNHIP_BL_ARGS);
    if (K <= 48) return launch_batch_levels<C, 12>(GNNHIP_BL_ARGS);
    return launch_batch_levels<C, 16>(GNNHIP_BL_ARGS);
#undef GNNHIP_BL_ARGS
}

constexpr int kTwoStepMeanDegree = 12;           // denser matrices take the SpMM

}  // namespace

// msg and the last level's h of a batch of small graphs.  work: at least batch_levels_work_ints(B) ints, 16-byte aligned.  *refused: the
// device word that says (1) that the batch is none and the outputs have to be formed by the level-by-level route.
// GNNHIP_EUNSUPPORTED (nothing launched): sizes that this route does not take.
size_t batch_levels_work_ints(int B) { return kOrderRec + bin_ints(B); }

int batch_levels_dispatch(int N, int B, int K, int C, int L, long long nnz, const int* a_row_ptr, const int* a_col_idx, const float* a_val,
                          const int* s_row_ptr, const float* X, const float* Wn2l, const float* Wc, float* msg, float* h_out, int* work,
                          const int** refused, hipStream_t s)
{
    // What the levels but the first save is reading h and msg and writing h.  Below these products the launches of both routes cost more
    // than that (hidden 64, 35,000 nodes: two levels 52 us against 48, three 59 against 62; hidden 32, 73,000 nodes: one level 35.6 against
    // 35.2, two 42.9 against 45.6).
    const bool enough = (long long)(L - 1) * N * C >= (C == 16 ? 12000000 : 4000000) && N >= 32768;
    if (!enough || nnz >= kTwoStepMeanDegree * (long long)N || (long long)N > 96ll * B || K < 2 || K > 64 || !(C == 16 || C == 32 || C == 64))
        return GNNHIP_EUNSUPPORTED;
    int* word = work;
    int* bins = work + kOrderRec;
    hipLaunchKernelGGL((graph_bins_kernel<true>), dim3(ceil_div_u((size_t)B, kBinBlock)), dim3(kBinBlock), 0, s, B, kRows, a_row_ptr, s_row_ptr,
                       bins, N, word);
    GNNHIP_LAUNCH_CHECK("graph_bins");
    *refused = word;
#define GNNHIP_BL_ARGS N, B, K, L, a_row_ptr, a_col_idx, a_val, X, Wn2l, Wc, msg, h_out, bins, word, s
    switch (C) {
    case 16: return batch_levels_c<16>(GNNHIP_BL_ARGS);
    case 32: return batch_levels_c<32>(GNNHIP_BL_ARGS);
    default: return batch_levels_c<64>(GNNHIP_BL_ARGS);
    }
#undef GNNHIP_BL_ARGS
}

}  // namespace gnnhip
