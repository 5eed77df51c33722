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
// (0.6 GB), and the pooled rows S h are added up from LDS as well, where enough is read less for the launch that this takes (the
// readout's own pass over h: 71 us of 444).  880,690 nodes, four levels, the whole forward: hidden 64 768 -> 403 us, hidden 32
// 419 -> 226; a level more 158 -> 55 and 87 -> 30.
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
// 1.16e-11 of the terms' magnitudes after four levels, level by level 2.42e-11.  Counted there, vector instructions
// take 40 % of the cycles (about 330 per 16 rows and level: 64 sum the first four entries, 104 split the rows), the matrix pipes 28 %, the LDS 27 %,
// a quarter of that bank conflicts, and memory moves 1.6 TB/s: no unit bounds that kernel but that it has two wavefronts per SIMD (247 registers), which
// meet at two barriers per level and wait 41 % of their time.  What a bin reads is asked for while the last level of the bin before it ends (428 us without).
//
// Hidden sizes from 17 to 112 without kernels of their own take the next multiple of 16, with zeros behind the last column.  msg comes from
// memory (the general input stage: 12 us of 91 at 44,000 nodes, hidden 100, and the launch) only where W_n2l does not fit or K is 1 or
// more than 64.  Above 64 W lies in LDS in all three pieces (86 KB at 112) and a workgroup fills a compute unit:
// its wavefronts wait for the same things at the same time, and a level of 16 rows reads all of W.  44,000 nodes, hidden 100, 3.8
// entries per row: a level 28 -> 15 us, the forward of three 111 -> 82; 176,000 nodes, four levels 416 -> 245; error against float64
// 6.7e-11, was 1.4e-10.  Above 112 columns W and the rows of 128 nodes do not fit the LDS together.  Tried there: the wavefronts share
// the columns, as in level_wide_split.hip, and the rows are put into pieces in place between two barriers: 7.5 us for a bin of 112
// nodes and a level at hidden 128, where the level-by-level route takes as long, and at hidden 256, where 64 nodes fit, 1.5 times that.
#include <type_traits>

#include "bf16_split.h"
#include "columns.h"
#include "graph_bins.h"

namespace gnnhip {

// hub.hip
int hub_count_with_bins(int m, int n, long long nnz, const int* row_ptr, const BinsArgs& bins, hipStream_t s, bool* counted);

namespace {

constexpr int kRows = 128;                       // nodes of a bin
constexpr int kEdgeCap = 1024;                   // entries of a bin kept in LDS; those of a bin with more are read from memory in every level
constexpr int kDirect = 4;                       // entries per row whose place and weight stay in registers

// CP: hidden size, or the next multiple of 16 that has a kernel.  TPW: tiles of 16 rows per wavefront.  MINW: wavefronts per SIMD.
// PIECES: products from bf16 pieces; WREG: the first two pieces of W in registers, else all three in LDS
template <int CP> struct BatchShape { static constexpr int TPW = 1, MINW = 2; static constexpr bool PIECES = true, WREG = false; };
template <> struct BatchShape<16> { static constexpr int TPW = 1, MINW = 6; static constexpr bool PIECES = false, WREG = true; };
template <> struct BatchShape<32> { static constexpr int TPW = 1, MINW = 4; static constexpr bool PIECES = false, WREG = true; };
template <> struct BatchShape<48> { static constexpr int TPW = 2, MINW = 2; static constexpr bool PIECES = true, WREG = true; };
template <> struct BatchShape<64> { static constexpr int TPW = 2, MINW = 2; static constexpr bool PIECES = true, WREG = true; };
template <int CP> constexpr int batch_waves() { return kRows / 16 / BatchShape<CP>::TPW; }
template <int CP> constexpr int w_lds_words()    // 128-bit words of W in LDS
{
    return !BatchShape<CP>::PIECES ? 0 : (CP / 4 + 7) / 8 * (CP / 16) * (BatchShape<CP>::WREG ? 1 : 3) * kWave;
}

template <int CP, int KSX>
constexpr size_t batch_lds_bytes()
{
    return sizeof(float) * (size_t)(kRows + 1) * (CP + 4) + sizeof(bf16_words4) * w_lds_words<CP>() + (BatchShape<CP>::PIECES ? sizeof(float) * CP : 0) +
           sizeof(float) * (size_t)(CP / 16) * KSX * kWave + sizeof(int2) * (kEdgeCap + kRows) + sizeof(int) * (kRows + 4 + kWave + 4);
}

// KSX: contraction steps of the input stage, K <= 4 KSX; 0: msg is there.  ODD: the hidden size is C <= CP, else CP
template <int CP, int KSX, bool ODD>
__global__ __launch_bounds__(batch_waves<CP>() * kWave, BatchShape<CP>::MINW) void s2v_batch_levels_kernel(
    int N, int B, int K, int hidden, int L, const int* __restrict__ a_row_ptr, const int* __restrict__ a_col_idx, const float* __restrict__ a_val,
    const int* __restrict__ s_row_ptr, const int* __restrict__ s_col_idx, const float* __restrict__ s_val, const float* __restrict__ X,
    const float* __restrict__ Wn2l, const float* __restrict__ Wc, float* __restrict__ msg, float* __restrict__ h_out,
    float* __restrict__ pool, const int* __restrict__ bins, int* __restrict__ refused)
{
    using Shape = BatchShape<CP>;
    constexpr int TPW = Shape::TPW, kWaves = batch_waves<CP>(), kBlock = kWaves * kWave;
    constexpr bool PIECES = Shape::PIECES, WREG = Shape::WREG, INPUT = KSX > 0;
    constexpr int KS = CP / 4;                   // columns of a lane, contraction steps of a level
    constexpr int KS2 = (KS + 7) / 8;            // contraction steps of a level in pieces
    constexpr int NJB = CP / 16;                 // output blocks of 16 columns
    constexpr int LD = CP + 4;
    const int C = ODD ? hidden : CP;
    const bool pooled = CP > 16 && pool;
    static_assert(!PIECES || !WREG || KS2 == 2, "two sums of opposite signs");
    extern __shared__ float4 smem4[];
    float* hbuf = reinterpret_cast<float*>(smem4);                         // [kRows + 1][LD], the last row zeros
    bf16_words4* w_lds = reinterpret_cast<bf16_words4*>(hbuf + (kRows + 1) * LD);          // W in pieces, [KS2][NJB][3][lane], or the third ones
    float* w_down = reinterpret_cast<float*>(w_lds + w_lds_words<CP>());   // [CP] a column's scale up over its scale
    float2* wn = reinterpret_cast<float2*>(w_down + (PIECES ? CP : 0));    // [NJB][KSX / 2][lane]
    int2* edges = reinterpret_cast<int2*>(wn + NJB * (KSX / 2) * kWave);   // [kEdgeCap] row offset, weight
    int2* members = edges + kEdgeCap;                                      // [kRows] row offset, weight: entries of S
    int* rp = reinterpret_cast<int*>(members + kRows);                     // [kRows + 1], from the bin's first entry on
    int* sp = rp + kRows + 4;                                              // [kWave + 1] the same of S
    __shared__ int stop;                         // another workgroup has come upon an entry that leaves its bin
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int row0 = 16 * TPW * wave + t;        // this lane's row of the bin in the wavefront's first tile
    const int out_col = KS * (t >> 2) + (t & 3); // column of W that a lane supplies to block jb: out_col + 4 jb
    // contraction steps of the input stage that are needed.  Steps 2 j and 2 j + 1 take k = 8 j + 2 q and the one behind it, so that a load of
    // a pair of columns by all lanes covers 32 consecutive bytes of 16 rows
    const int srt = 2 * ((K + 7) / 8);

    // a segment that was not packed (graph_bins.h): nothing is formed.  Every workgroup looks at all words, 64 graphs each, and does so ahead of
    // all else, so that a batch that is none costs little more than the launch (with W loaded and split first 8 to 10 us in a trace, so 3 to 4).
    // A forward that tries this for nothing, one graph of 600 nodes among others, four levels, without the attempt and with it: 30,000 graphs,
    // hidden 64 696 us and 706; 1,500, hidden 64 81 and 87; hidden 100 159 and 163; 600, hidden 100 97 and 104.  (Packing the segments of few graphs
    // in every workgroup here, without the bins' launch: as long for a batch that is none, 1 to 16 % longer for one that is taken.  The input stage
    // of a refused batch here: 15 us where its own kernel takes 8.)
    bool unpacked = false;
    for (int i = tid; i < (B + kWave - 1) / kWave; i += kBlock) unpacked |= reinterpret_cast<const unsigned long long*>(bins)[i] == 0;
    if (__syncthreads_or(unpacked)) {
        if (tid == 0) *refused = 1;
        return;
    }
    BinFinder finder(B, bins);
    int at = finder.find((int)blockIdx.x);

    // W as the operand of the matrix instructions, zeros past its last row and column.  fp32: wf[jb][s] = W[KS q + s][out_col + 4 jb]; in
    // pieces: of W[KS q + 8 s + 0..7].  The matrix instructions on bf16 round towards minus infinity: in registers, the second step is
    // negated and summed apart, so that the drifts cancel; in LDS, every other block of columns is negated, so that there is no drift
    // from level to level.
    float wf[PIECES ? 1 : NJB][PIECES ? 1 : KS];
    bf16_words4 wp[PIECES && WREG ? KS2 : 1][PIECES && WREG ? NJB : 1][2];
    bool any_down = false;                       // a column of W is scaled down (bf16_split.h): uniform
    auto w_at = [&](int k, int jb) {             // k: of the lane's
        const int row = KS * q + k, col = out_col + 4 * jb;
        return !ODD || (row < C && col < C) ? Wc[(size_t)row * C + col] : 0.f;
    };
    auto put_w = [&](int jb, const float (&w)[8 * KS2]) {
        float largest = 0.f;
#pragma unroll
        for (int k = 0; k < KS; k += 2) largest = split_max(largest, w[k], w[k + 1]);
        const unsigned long long large = __ballot(largest >= kSplitLarge);
        const bool down = (large >> t) & 0x0001000100010001ull;            // in any quarter of the column
        any_down |= large != 0;
        const float scale = down ? kSplitDown : kSplitUp;
        if (q == 0) w_down[out_col + 4 * jb] = down ? kSplitUp / kSplitDown : 1.f;
#pragma unroll
        for (int s = 0; s < KS2; ++s) {
            bf16_words4 w3[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                unsigned p[3];
                bf16_split2(w[8 * s + 2 * i] * scale, w[8 * s + 2 * i + 1] * scale, down, p);
                const unsigned sign = (WREG ? s : jb) % 2 ? 0x80008000u : 0u;
#pragma unroll
                for (int j = 0; j < 3; ++j) w3[j][i] = p[j] ^ sign;
            }
            if constexpr (WREG) {
                wp[s][jb][0] = w3[0]; wp[s][jb][1] = w3[1];
                if (wave == 0) w_lds[(s * NJB + jb) * kWave + lane] = w3[2];
            } else {
#pragma unroll
                for (int j = 0; j < 3; ++j) w_lds[((s * NJB + jb) * 3 + j) * kWave + lane] = w3[j];
            }
        }
    };
    if constexpr (PIECES) {
#pragma unroll
        for (int j0 = 0; j0 < (WREG ? NJB : (NJB + kWaves - 1) / kWaves); ++j0) {
            const int jb = WREG ? j0 : j0 * kWaves + wave;
            if (jb >= NJB) continue;             // uniform
            float w[8 * KS2];
#pragma unroll
            for (int k = 0; k < 8 * KS2; ++k) w[k] = k < KS ? w_at(k, jb) : 0.f;
            put_w(jb, w);
        }
    } else {
#pragma unroll
        for (int jb = 0; jb < NJB; ++jb)
#pragma unroll
            for (int s = 0; s < KS; ++s) wf[jb][s] = w_at(s, jb);
    }
    if constexpr (INPUT) {
        for (int i = wave; i < NJB * (KSX / 2); i += kWaves) {
            const int jb = i / (KSX / 2), k = 8 * (i % (KSX / 2)) + 2 * q;
            const bool in = !ODD || out_col + 4 * jb < C;
            wn[i * kWave + lane] = make_float2(in && k < K ? Wn2l[(size_t)k * C + out_col + 4 * jb] : 0.f,
                                               in && k + 1 < K ? Wn2l[(size_t)(k + 1) * C + out_col + 4 * jb] : 0.f);
        }
    }
    if (tid < LD) hbuf[kRows * LD + tid] = 0.f;
    if (tid == 0) stop = 0;
    any_down = __syncthreads_or(any_down);

    // ---- what a bin needs from memory, asked for together and a bin ahead
    struct Bin { int node0, n, e0, ne, g0, ng; };
    auto record = [&](int at) {
        const int* rec = bins + bin_words_ints(B) + (size_t)max(at, 0) * kOrderRec;
        const int4 r = *reinterpret_cast<const int4*>(rec);
        const int2 r2 = *reinterpret_cast<const int2*>(rec + 4);
        return at < 0 ? Bin{0, 0, 0, 0, 0, 0} : Bin{r.y, r.z, r.w, max(r2.x - r.w, 0), r.x, r2.y};
    };
    constexpr int kEdgesEach = kEdgeCap / kBlock;
    float x[TPW][INPUT ? KSX : 1], e_val[kEdgesEach];
    float4 mx[TPW][INPUT ? 1 : NJB];             // rows of msg where they are there already
    int e_col[kEdgesEach], rp_v, sp_v, s_col;
    float s_w;
    auto ask = [&](const Bin& b) {
        // (every register is written whatever the bin is, or the old values would have to be kept through the levels)
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            const size_t at_row = (size_t)min(b.node0 + min(row0 + 16 * i, max(b.n - 1, 0)), N - 1);
            if constexpr (!INPUT) {
                const float* mr = msg + at_row * C;
#pragma unroll
                for (int jb = 0; jb < NJB; ++jb) {
                    const int col = KS * q + 4 * jb;
                    mx[i][jb] = f4_zero();
                    if (col + 4 <= C) {
                        mx[i][jb] = ColsLoose::load(mr + col);
                    } else {
                        if (col < C) mx[i][jb].x = mr[col];
                        if (col + 1 < C) mx[i][jb].y = mr[col + 1];
                        if (col + 2 < C) mx[i][jb].z = mr[col + 2];
                    }
                }
            }
            const float* xr = X + at_row * K;
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
        sp_v = pooled ? s_row_ptr[b.g0 + min(tid, b.ng)] : 0;
        s_col = pooled && tid < b.n ? s_col_idx[b.node0 + tid] : b.node0;    // (graph g's entries of S are numbered as its nodes are)
        s_w = pooled && tid < b.n ? s_val[b.node0 + tid] : 0.f;
        const int in_lds = b.ne <= kEdgeCap ? b.ne : 0;
#pragma unroll
        for (int u = 0; u < kEdgesEach; ++u) {
            const int e = tid + u * kBlock;
            e_col[u] = e < in_lds ? a_col_idx[b.e0 + e] : 0;
            e_val[u] = e < in_lds ? a_val[b.e0 + e] : 0.f;
        }
    };
    auto mask = [&](float4 (&v)[NJB]) {          // ODD: zeros past the last column (in the last quarter, q = 3)
        if (C == CP) return;
#pragma unroll
        for (int jb = NJB > 4 ? NJB - 4 : 0; jb < NJB; ++jb) {
            const int col = KS * q + 4 * jb;
            v[jb].x = col < C ? v[jb].x : 0.f;
            v[jb].y = col + 1 < C ? v[jb].y : 0.f;
            v[jb].z = col + 2 < C ? v[jb].z : 0.f;
            v[jb].w = col + 3 < C ? v[jb].w : 0.f;
        }
    };
    Bin cur = record(at), next;
    bool more = at >= 0;                         // there is a bin `cur`
    ask(cur);

    for (int bin = blockIdx.x; more && !stop; bin += gridDim.x) {
        // (the same in all wavefronts: stop is written between two barriers that this test does not lie between)
        const int node0 = cur.node0, n = cur.n, e0 = cur.e0, ne = cur.ne, g0 = cur.g0, ng = cur.ng;
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
        at = finder.find(bin + (int)gridDim.x);
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
            for (int jb = 0; jb < NJB; ++jb) {
                m[i][jb] = f4_zero();
                if (row0 + 16 * i < n) m[i][jb] = INPUT ? make_float4(acc[jb][0], acc[jb][1], acc[jb][2], acc[jb][3]) : mx[i][INPUT ? 0 : jb];
            }
            if constexpr (ODD && INPUT) mask(m[i]);
        }
        __syncthreads();                         // the last bin's rows have left hbuf; rp and edges are there
        if (pooled && tid < n) {
            const int c = s_col - node0;
            if (c < 0 || c >= n) *refused = 1;
            members[tid] = make_int2(min(max(c, 0), n - 1) * LD, __float_as_int(s_w));
        }
        if (pooled && tid <= ng) sp[tid] = sp_v - node0;
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
        // (what follows from these is not kept through the levels)
        auto lane_now = [&]() { int l = lane; asm("" : "+v"(l)); return l; };
        auto tid_now = [&]() { int l = tid; asm("" : "+v"(l)); return l; };
        // the bin's rows as they lie in memory: whole lines
        auto copy_out = [&](float* dst) {
            const int tid = tid_now();
            if constexpr (!ODD) {
                for (int i = tid; i < n * KS; i += kBlock)
                    *reinterpret_cast<float4*>(dst + (size_t)node0 * C + 4 * i) = *reinterpret_cast<const float4*>(hbuf + (i / KS) * LD + 4 * (i % KS));
            } else {
                constexpr int G = KS <= 4 ? 4 : KS <= 8 ? 8 : KS <= 16 ? 16 : 32;      // lanes per row
                const int col = 4 * (tid % G);
                if (col < C) {
                    for (int r = tid / G; r < n; r += kBlock / G) {
                        const float4 v = *reinterpret_cast<const float4*>(hbuf + r * LD + col);
                        float* d = dst + (size_t)(node0 + r) * C + col;
                        if (col + 4 <= C) {
                            ColsLoose::store(d, v);
                        } else {
                            d[0] = v.x;
                            if (col + 1 < C) d[1] = v.y;
                            if (col + 2 < C) d[2] = v.z;
                        }
                    }
                }
            }
        };
        if (INPUT) copy_out(msg);
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
                        if (kRelu) r = PIECES ? relu_max4(r) : relu_ref4(r);
                        agg[k] += w * r.x; agg[k + 1] += w * r.y; agg[k + 2] += w * r.z; agg[k + 3] += w * r.w;
                    }
                };
                if (staged) {
#pragma unroll
                    for (int u = 0; u < kDirect; ++u) add(g_off[i][u], g_w[i][u]);
                    int e = g_st[i] + kDirect;
                    if (e < g_en[i]) {
                        int2 ed = edges[e];
                        do {                     // the next entry is on its way while this one's row is added
                            const int2 now = ed;
                            ed = edges[min(++e, kEdgeCap - 1)];
                            add(now.x + KS * q, __int_as_float(now.y));
                        } while (e < g_en[i]);
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
                                unsigned w[3] = {0, 0, 0};
                                if (8 * s + 2 * u < KS) bf16_split2(agg[8 * s + 2 * u] * scale, agg[8 * s + 2 * u + 1] * scale, down, w);
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
                    // The corrections come ahead of the products of the first pieces: with W in registers in the same sum, one per step, the second of
                    // the other sign; with W in LDS in a sum of their own
                    mfma_f4 acc[2][NJB];
#pragma unroll
                    for (int jb = 0; jb < NJB; ++jb) acc[0][jb] = acc[1][jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (WREG) {
                        auto products = [&](int w, int x) {
#pragma unroll
                            for (int s = 0; s < KS2; ++s)
#pragma unroll
                                for (int jb = 0; jb < NJB; ++jb)
                                    acc[s][jb] = mfma_bf16(w == 2 ? w_lds[(s * NJB + jb) * kWave + lane] : wp[s][jb][w < 2 ? w : 0], p[s][x], acc[s][jb]);
                        };
                        products(2, 0); products(0, 2); products(1, 1); products(1, 0); products(0, 1); products(0, 0);
                    } else {
#pragma unroll
                        for (int s = 0; s < KS2; ++s) {
                            // a few blocks at a time, so that no product waits for the sum of the one before it
                            constexpr int kGroup = 4;
#pragma unroll
                            for (int j0 = 0; j0 < NJB; j0 += kGroup) {
                                bf16_words4 w[kGroup][3];
#pragma unroll
                                for (int j = 0; j < kGroup; ++j)
#pragma unroll
                                    for (int i = 0; i < 3; ++i)
                                        if (j0 + j < NJB) w[j][i] = w_lds[((s * NJB + j0 + j) * 3 + i) * kWave + lane];
                                auto products = [&](int sum, int i, int x) {
#pragma unroll
                                    for (int j = 0; j < kGroup; ++j)
                                        if (j0 + j < NJB) acc[sum][j0 + j] = mfma_bf16(w[j][i], p[s][x], acc[sum][j0 + j]);
                                };
                                products(1, 2, 0); products(0, 0, 0); products(1, 0, 2); products(1, 1, 1); products(1, 1, 0); products(1, 0, 1);
                            }
                        }
                    }
#pragma unroll
                    for (int jb = 0; jb < NJB; ++jb) {
                        const float b = WREG || jb % 2 == 0 ? back : -back;
                        float4 f = make_float4(b, b, b, b);
                        if (any_down) {
                            const float4 d = *reinterpret_cast<const float4*>(w_down + KS * q + 4 * jb);
                            f.x *= d.x; f.y *= d.y; f.z *= d.z; f.w *= d.w;
                        }
                        const mfma_f4 r = WREG ? acc[0][jb] - acc[1][jb] : acc[0][jb] + acc[1][jb];
                        v[i][jb] = relu_max4(make_float4(fmaf(r[0], f.x, m[i][jb].x), fmaf(r[1], f.y, m[i][jb].y), fmaf(r[2], f.z, m[i][jb].z),
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
            if constexpr (ODD) {                 // columns past the last stay zero whatever the others are
#pragma unroll
                for (int i = 0; i < TPW; ++i)
                    if (i < tiles) mask(v[i]);
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
        level(std::true_type(), std::false_type());      // (L >= 2)
        for (int lv = 2; lv < L; ++lv) level(std::false_type(), std::false_type());
        level(std::false_type(), std::true_type());
        copy_out(h_out);
        // pool = S h: a wavefront per graph, kLanes lanes per row
        if (pooled) {
            constexpr int kLanes = KS <= 4 ? 4 : KS <= 8 ? 8 : KS <= 16 ? 16 : 32, kApart = kWave / kLanes;
            const int l = lane_now();
            const int col = 4 * (l % kLanes);
            for (int g = wave; g < ng; g += kWaves) {
                const int end = min(sp[g + 1], n);
                float4 sum = f4_zero();
                for (int r = sp[g] + l / kLanes; r < end; r += 4 * kApart) {
                    int2 of[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        of[u] = members[min(r + u * kApart, kRows - 1)];
                        if (r + u * kApart >= end) of[u] = make_int2(kRows * LD, 0);
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (kLanes == KS || col < CP) f4_fma(sum, __int_as_float(of[u].y), *reinterpret_cast<const float4*>(hbuf + of[u].x + col));
                }
#pragma unroll
                for (int d = kLanes; d < kWave; d <<= 1)
                    sum = ColsWide::add(sum, make_float4(__shfl_xor(sum.x, d, kWave), __shfl_xor(sum.y, d, kWave), __shfl_xor(sum.z, d, kWave),
                                                         __shfl_xor(sum.w, d, kWave)));
                float* to = pool + (size_t)(g0 + g) * C + col;
                if (l < kLanes && col < C) {
                    if (!ODD) {
                        *reinterpret_cast<float4*>(to) = sum;
                    } else if (col + 4 <= C) {
                        ColsLoose::store(to, sum);
                    } else {
                        to[0] = sum.x;
                        if (col + 1 < C) to[1] = sum.y;
                        if (col + 2 < C) to[2] = sum.z;
                    }
                }
            }
        }
        cur = next;
    }
}

template <int CP, int KSX, bool ODD>
int launch_batch_levels(int N, int B, int K, int C, int L, const int* a_row_ptr, const int* a_col_idx, const float* a_val, const int* s_row_ptr,
                        const int* s_col_idx, const float* s_val, const float* X, const float* Wn2l, const float* Wc, float* msg, float* h_out,
                        float* pool, const int* bins, int* refused, int cap, hipStream_t s)
{
    constexpr size_t smem = batch_lds_bytes<CP, KSX>();
    constexpr int kWaves = batch_waves<CP>();
    static_assert(smem * (BatchShape<CP>::MINW * 4 / kWaves) <= 160 * 1024, "workgroups share the LDS of a compute unit");
    static LdsLimit lds_limit;
    GNNHIP_HIP(lds_limit.raise(reinterpret_cast<const void*>(&s2v_batch_levels_kernel<CP, KSX, ODD>), smem));
    // two neighbouring bins hold more than cap nodes together, and every 64 graphs may leave one bin short
    long long most = 2ll * N / cap + (B + kWave - 1) / kWave + 1;
    if (most > B) most = B;
    const long long resident = (long long)kNumCU * (BatchShape<CP>::MINW * 4 / kWaves);
    const unsigned grid = (unsigned)(most < resident ? most : resident);
    hipLaunchKernelGGL((s2v_batch_levels_kernel<CP, KSX, ODD>), dim3(grid), dim3(kWaves * kWave), smem, s, N, B, K, C, L, a_row_ptr, a_col_idx, a_val,
                       s_row_ptr, s_col_idx, s_val, X, Wn2l, Wc, msg, h_out, pool, bins, refused);
    GNNHIP_LAUNCH_CHECK("s2v_batch_levels");
    return GNNHIP_OK;
}

constexpr int kTwoStepMeanDegree = 12;           // denser matrices take the SpMM

}  // namespace

size_t batch_levels_work_ints(int B) { return bin_ints(B); }

// whether the levels' launch forms the pooled rows too: the readout reads h otherwise, but needs a launch less (hidden 100, 44,000
// nodes 93 us, 96 with them, 88,000 135 and 138, 176,000 218 and 212, 352,000 405 and 390; hidden 64 of 9 features, 73,000 nodes 73 and 70; hidden
// 50, 88,000 nodes 87 and 85; hidden 32, 73,000 nodes 51 and 50, 294,000 82 and 78; hidden 16 587,000 nodes 92 and 92, of 60 features 142 and 146)
bool batch_levels_with_pool(int N, int C) { return C > 16 && (long long)N * C >= (C > 64 ? 12000000 : 4000000); }

// Whether a forward tries the one launch, and how.
BatchRoute batch_levels_route(int N, int B, int K, int C, int L, long long nnz)
{
    BatchRoute route;
    // (past 96 columns there is no more LDS for W_n2l of many rows)
    const bool input = K >= 2 && C >= 16 && (K <= 16 ? C <= 112 : K <= 64 && C <= 96);
    // What the levels but the first save is reading h and msg and writing h, and, where the level-by-level kernels are those of any size, most
    // of a level.  Below these products the launches of both routes cost more than that.  Forwards, level by level and so:
    //     hidden 66     6,755 nodes, three levels (0.9 M) 39 us and 39, four 47 and 43; 14,102, two (0.9 M) 36 and 35, five 67 and 49
    //            96     20,564, two (2 M) 49 and 37, four 81 and 48;  100 of 38 features, where the input is a launch: 20,564, two (2.1 M) 52 and 52
    //            56     14,102, five (3.2 M) 52 and 54; 20,564, four (3.5 M) 51 and 50;  50: 26,440, four (4 M) 56 and 50; 52,870, three 80 and 63
    //            20     26,440, three (1.1 M) 32 and 33, four 38 and 36; 52,870, three (2.1 M) 54 and 46
    //            64     26,440, three (3.4 M) 41 and 42, four 50 and 48;  32: 52,870, three (3.4 M) 48 and 44
    //            16     73,432, four (3.5 M) 53 and 51 or, of 38 features, 58 and 50; 52,870, five (3.4 M) 57 and 64
    // Up to kLevelTileMaxRows nodes hidden 16, 32 and 64 have level_tile.hip, up to kFewRows the others the kernel of few rows: neither has a gated variant.
    const bool own = C == 16 || C == 32 || C == 64;
    // At hidden 16 a bin whose entries do not fit the LDS costs more than it saves (three levels, 300,573 nodes: 9 entries per row 95 us and 94, 10 97 and 107,
    // 11.5 105 and 122; 587,454 in graphs of 10 to 110, 8.4 133 and 118, 10 155 and 179)
    const long long dense = C == 16 ? 9 : kTwoStepMeanDegree;
    if (nnz >= dense * N || (long long)N > 96ll * B || C < 16 || C > 112) return route;
    // Bins of fewer nodes where they fill the rounds of workgroups better: a round takes its tiles and about two more (start, barriers).
    // The host knows the totals only: a bin wastes about 0.6 of a mean graph (half of the graph that no longer fits, and large ones are met more often), and every
    // 64 graphs about half a bin.
    const int slots = kNumCU * (C <= 16 ? 3 : C <= 64 ? 2 : 1);
    long long rounds = 1;
    double best = 0.0;
    for (int c = kRows; c >= 64; c -= 16) {
        const double fill = (double)c - 0.6 * (double)N / (double)B;
        const double nbins = (double)N / (fill > 16.0 ? fill : 16.0) + (double)B / 128.0;
        const long long r = (long long)(nbins / slots) + 1;
        const double cost = (double)r * (2.0 + c / 16);
        if (c == kRows || cost < best) { best = cost; route.cap = c; rounds = r; }
    }
    // Up to 128 rows per compute unit the level-by-level kernels are at their best, and bins that need a second round of workgroups lose to them with few levels (28,000
    // nodes of 38 features, hidden 72, two levels 44.8 us and 48.3; hidden 100 of 7, two 53.4 and 54.4; of 38, three 77.6 and 79.0); so does hidden 64 in one
    // round (28,000, four levels 44.9 and 48.3, five 58 and 56), which meets a second one below 65,536 nodes, where they have not yet slowed down again
    // (60,000, three 64.3 and 65.8, four 76.3 and 78.1, five 100 and 95)
    const bool few = N <= 128 * kNumCU, again = rounds > 1;
    long long least;
    if (C <= 32) least = C == 16 ? 5000000 : C == 32 ? 3000000 : 1500000;
    else if (C < 64) least = L == 2 || (L == 3 && few) ? 4100000 : 3600000;        // (hidden 56, 70,000 nodes, two levels 71.6 us and 74.9, 75,000 73 and 68)
    else if (C == 64) least = few ? 6300000 : again && N < 65536 ? 12000000 : 4000000;
    else if (!input) least = few && again ? 7500000 : 4000000;
    else least = few && again ? 3700000 : C <= 96 ? 1500000 : 1800000;
    // Graphs of more than half a bin leave much of it empty (all of 65 nodes, hidden 64 of 38 features: 52,000, five levels 86 us and 101, 150,000, two 86 and 100, three
    // 114 and 119, 300,000, two 146 and 158; hidden 56, 90,000, two 69 and 81)
    if (2ll * N > (long long)kRows * B) least *= L == 2 ? 6 : 3;
    if ((long long)(L - 1) * N * C < least || N <= (own ? kLevelTileMaxRows : C > 32 && C < 64 ? 64 * kNumCU : kFewRows)) return route;
    route.take = true;
    route.input = input;
    return route;
}

// The launch ahead of the levels' one: the bins.  work: at least batch_levels_work_ints(B) ints, 16-byte aligned, free once the levels'
// launch is done.  planned: A has a kept plan, which counts the long rows of A once and for all; else *counted: the levels' first hub_prepass may
// reuse the plan of them that the call has left in the stream's scratch.
int batch_levels_bins(const BatchRoute& route, int N, int B, int C, long long nnz, const int* a_row_ptr, const int* s_row_ptr, int* work, int* refused,
                      bool planned, bool* counted, hipStream_t s)
{
    const BinsArgs bins{B, route.cap, a_row_ptr, s_row_ptr, work, N, kRows, refused};
    if (!planned) return hub_count_with_bins(N, C, nnz, a_row_ptr, bins, s, counted);
    hipLaunchKernelGGL((graph_bins_kernel<true>), dim3(ceil_div_u((size_t)B, kBinBlock)), dim3(kBinBlock), 0, s, bins);
    GNNHIP_LAUNCH_CHECK("graph_bins");
    return GNNHIP_OK;
}

// The last level's h and, unless pool is null, the pooled rows (and msg) of a batch of small graphs.  bins: as batch_levels_bins left them.  *refused: the device
// word that says (1) that the batch is none and the outputs have to be formed by the level-by-level route.  L >= 2 (batch_levels_route).
int batch_levels_dispatch(const BatchRoute& route, int N, int B, int K, int C, int L, const int* a_row_ptr, const int* a_col_idx, const float* a_val,
                          const int* s_row_ptr, const int* s_col_idx, const float* s_val, const float* X, const float* Wn2l, const float* Wc,
                          float* msg, float* h_out, float* pool, const int* bins, int* refused, hipStream_t s)
{
    const bool input = route.input;
    const int cap = route.cap;
#define GNNHIP_BL(CP, KSX, ODD) launch_batch_levels<CP, KSX, ODD>(N, B, K, C, L, a_row_ptr, a_col_idx, a_val, s_row_ptr, s_col_idx, s_val, X, Wn2l, Wc, msg, h_out, \
                                                pool, bins, refused, cap, s)
    if (input && (C == 16 || C == 32 || C == 64)) {
#define GNNHIP_BL_K(CP) (K <= 16 ? GNNHIP_BL(CP, 4, false) : K <= 32 ? GNNHIP_BL(CP, 8, false) : K <= 48 ? GNNHIP_BL(CP, 12, false) : GNNHIP_BL(CP, 16, false))
        return C == 16 ? GNNHIP_BL_K(16) : C == 32 ? GNNHIP_BL_K(32) : GNNHIP_BL_K(64);
#undef GNNHIP_BL_K
    }
#define GNNHIP_BL_K(CP) (!input ? GNNHIP_BL(CP, 0, true) : K <= 16 ? GNNHIP_BL(CP, 4, true) : GNNHIP_BL(CP, 16, true))
    switch ((C + 15) / 16) {
    case 1: return GNNHIP_BL(16, 0, true);
    case 2: return GNNHIP_BL_K(32);
    case 3: return GNNHIP_BL_K(48);
    case 4: return GNNHIP_BL_K(64);
    case 5: return GNNHIP_BL_K(80);
    case 6: return GNNHIP_BL_K(96);
    default: return input ? GNNHIP_BL(112, 4, true) : GNNHIP_BL(112, 0, true);
    }
#undef GNNHIP_BL_K
#undef GNNHIP_BL
}

}  // namespace gnnhip
