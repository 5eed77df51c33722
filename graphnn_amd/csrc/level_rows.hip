// Mean-field level and its input stage for hidden sizes that no tuned kernel covers (4 <= C <= 256):
//
//   level      h_out = ReLU((A * h_in) * W + bias + msg)
//   backward   u = A' * dz ; g_prev = u * W^T, zeroed where gate <= 0 ; acc += g_prev
//   dense      out = X * W (+ bias + msg, ReLU), and a second output ReLU(out)
//
// as one launch each, instead of an SpMM, a GEMM and an element-wise pass over N x C.  Measured at 48,750 nodes, hidden 100,
// 4.8 entries per row: 41 -> 31 us per level and 28 -> 11 us for the input stage; 130,000 nodes, hidden 199: 400 -> 190 us.
// The FP32 matrix cores bound the wide sizes (11 of the 31 us, 115 of the 190), memory the narrow ones.
//
// A workgroup takes R = 16 RT consecutive rows:
//   1. the rows of the left operand are put into LDS [R][KP + 4], KP = their width rounded up to 16, zeros behind it.  Gathered
//      rows: the tile's CSR entries, which lie next to each other, are copied to LDS first when there are at most kStaged,
//      then a group of G lanes (a power of two, 4 G >= width) sums a row, eight gathers in flight, entries in order;
//   2. the four wavefronts share the 16-column blocks of the product, up to NB each, all R rows: v_mfma_f32_16x16x4_f32, W
//      straight from L2 one step of 16 k ahead (40 KB per tile at hidden 100 against 128 KB of gathered rows).  Sharing out
//      the blocks of the last, uneven round row by row of blocks was tried: the extra loads of W cost more (179 -> 214 us at
//      390,000 nodes, hidden 85);
//   3. the product goes back through the same LDS, rows packed at their own width, so that what follows (msg, gate, sums,
//      ReLU, stores) walks flat words of four floats whatever the width: the R rows of a tile are contiguous.
// Sums have the order of the row-group SpMM and of the GEMM tile kernel, so every bit is theirs.
//
// Rows of more than kHubThreshold entries come from the balanced pass (hub.hip) where it runs, as in the SpMM; elsewhere rows
// longer than kLongRow are summed by the whole workgroup.
#include "columns.h"
#include "buffer_addr.h"

namespace gnnhip {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kStaged = 1024;             // CSR entries of a tile copied to LDS (8 KB)
constexpr int kLongRow = 2048;
constexpr int kMaxWidth = 256;            // of the left operand's rows and of the product's
constexpr int kFlight = 8;

struct RowsArgs {
    int N, K, n;                          // rows, width of the left operand, width of the product
    const int *row_ptr, *col_idx;         // gathered left operand (A * x); null row_ptr: x itself
    const float *val, *x, *W;
    const float *bias, *msg, *gate;       // msg: added; gate: product zeroed where gate <= 0
    float *agg_out, *out, *relu_out, *acc;   // agg_out: the left operand's rows; relu_out: ReLU(out); acc: += out
    int relu, relu_in;
    unsigned k_magic;                     // ceil(2^32 / K)
    HubPlan hubs;
    const int* launch_gate;               // see gated_off
};

// GATHER: the left operand is A * x.  WT: the product is with W^T.  MINW: wavefronts per SIMD the registers leave room for.
template <int RT, int NB, int MINW, bool GATHER, bool WT, bool GATED>
__global__ __launch_bounds__(kBlock, MINW) void s2v_rows_kernel(RowsArgs a)
{
    if (gated_off<GATED>(a.launch_gate)) return;
    using V = ColsLoose;
    constexpr int R = 16 * RT;
    extern __shared__ float4 smem4[];
    __shared__ int rp[R + 1];
    __shared__ float4 shared4[GATHER ? kStaged / 2 : 1];       // the tile's entries, then the sums of its long rows
    int2* staged = reinterpret_cast<int2*>(shared4);
    static_assert(kStaged / 2 >= kBlock, "a word per lane");
    __shared__ int long_row[GATHER ? R : 1];
    __shared__ int long_count;
    float* tile = reinterpret_cast<float*>(smem4);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int q = lane >> 4, t = lane & 15;
    const int K = a.K, n = a.n;
    const int KP = (K + 15) & ~15, LD = KP + 4;
    const long long row0 = (long long)blockIdx.x * R;
    const int rows = (int)min((long long)R, (long long)a.N - row0);

    // ---- W of step k0 for this wavefront's column blocks: wf[b][s] = W[k0 + 4 q + s][16 (wave + 4 b) + t], zero from k = K on
    const rsrc_t w_rsrc = make_rsrc(a.W, (unsigned)((size_t)K * n * 4));
    const int nb = wave < (n + 15) / 16 ? ((n + 15) / 16 - wave + kWaves - 1) / kWaves : 0;      // blocks of this wavefront
    auto load_w = [&](int k0, float (&wf)[NB][4]) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b >= nb) continue;                             // uniform
            const int col = 16 * (wave + kWaves * b) + t;
            if constexpr (WT) {
                // a lane's four k lie next to each other: one load instead of four, which matters where the rows of W are far apart
                // (backward at 48,750 nodes: hidden 120 47.8 -> 43.8 us, 160 109 -> 69, 199 105 -> 90)
                if (k0 + 16 <= K) {                            // uniform
                    const float4 w = V::load(a.W + (size_t)min(col, n - 1) * K + k0 + 4 * q);
                    wf[b][0] = w.x; wf[b][1] = w.y; wf[b][2] = w.z; wf[b][3] = w.w;
                    continue;
                }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int k = k0 + 4 * q + s;
                const int off = WT ? (col * K + k) * 4 : (k * n + col) * 4;       // a column past n: a word that is not stored
                wf[b][s] = buf_load_f(w_rsrc, k < K ? off : kBufPastEnd, 0);
            }
        }
    };
    float wf[NB][4];
    load_w(0, wf);

    // ---- 1. the left operand's rows
    if constexpr (GATHER) {
        if (tid <= R) rp[tid] = a.row_ptr[min(row0 + tid, (long long)a.N)];
        if (tid == 0) long_count = 0;
        for (int i = tid; i < R * 16; i += kBlock) {                    // the columns behind K
            const int c = KP - 16 + (i & 15);
            if (c >= K) tile[(i >> 4) * LD + c] = 0.f;
        }
        __syncthreads();
        const int lo = rp[0], hi = rp[R];
        const bool in_lds = hi - lo <= kStaged;
        if (in_lds) {
            for (int e = lo + tid; e < hi; e += kBlock) staged[e - lo] = make_int2(a.col_idx[e], __float_as_int(a.val[e]));
            __syncthreads();
        }
        const int units = (K + 3) / 4;
        const int logG = units <= 1 ? 0 : 32 - __builtin_clz((unsigned)(units - 1));
        const int G = 1 << logG, sub = tid & (G - 1), grp = tid >> logG, ngroups = kBlock >> logG;
        const bool live = sub < units;
        const int col0 = V::at(sub, K);
        auto add_row = [&](int start, int end, auto entry) {
            float4 sum = f4_zero();
            for (int base = start; base < end; base += kFlight) {
                int2 cv[kFlight];
                float4 x[kFlight];
#pragma unroll
                for (int u = 0; u < kFlight; ++u) cv[u] = base + u < end ? entry(base + u) : make_int2(0, 0);
#pragma unroll
                for (int u = 0; u < kFlight; ++u) x[u] = base + u < end && live ? V::load(a.x + (size_t)cv[u].x * K + col0) : f4_zero();
#pragma unroll
                for (int u = 0; u < kFlight; ++u)
                    if (base + u < end) f4_fma(sum, __int_as_float(cv[u].y), a.relu_in ? relu_ref4(x[u]) : x[u]);
            }
            return sum;
        };
        auto finish_row = [&](int r, const float4& sum) {
            if (!live) return;
            V::store(tile + r * LD + col0, sum);
            if (a.agg_out && r < rows) V::store(a.agg_out + (size_t)(row0 + r) * K + col0, sum);
        };
        for (int r = grp; r < R; r += ngroups) {
            const int start = rp[r], end = rp[r + 1];
            const int entries = end - start;
            int hub = -1;
            if (a.hubs.row_chunk && entries > kHubThreshold) hub = a.hubs.row_chunk[row0 + r];
            if (hub >= 0) {
                float4 sum = f4_zero();
                if (live) sum = V::axpby(f4_zero(), 1.f, hub_row_sum<V>(a.hubs.part + (size_t)hub * a.hubs.ld + col0, a.hubs.ld, entries, a.hubs.shift));
                finish_row(r, sum);
            } else if (entries > kLongRow) {
                if (sub == 0) long_row[atomicAdd(&long_count, 1)] = r;
            } else if (in_lds) {
                finish_row(r, add_row(start, end, [&](int e) { return staged[e - lo]; }));
            } else {
                finish_row(r, add_row(start, end, [&](int e) { return make_int2(a.col_idx[e], __float_as_int(a.val[e])); }));
            }
        }
        __syncthreads();
        const int nlong = long_count;
        for (int li = 0; li < nlong; ++li) {
            // the groups take entries grp, grp + ngroups, ...; their sums are added in group order
            const int r = long_row[li];
            const int start = rp[r], end = rp[r + 1];
            float4 sum = f4_zero();
            for (int e = start + grp; e < end; e += 4 * ngroups) {
                int c[4];
                float v[4];
                float4 x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const bool ok = e + u * ngroups < end;
                    c[u] = ok ? a.col_idx[e + u * ngroups] : 0;
                    v[u] = ok ? a.val[e + u * ngroups] : 0.f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) x[u] = e + u * ngroups < end && live ? V::load(a.x + (size_t)c[u] * K + col0) : f4_zero();
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (e + u * ngroups < end) f4_fma(sum, v[u], a.relu_in ? relu_ref4(x[u]) : x[u]);
            }
            shared4[tid] = sum;
            __syncthreads();
            if (grp == 0 && live) {
                float4 s = f4_zero();
                for (int g = 0; g < ngroups; ++g) s = V::add(s, shared4[g * G + sub]);
                V::store(tile + r * LD + col0, s);
                if (a.agg_out) V::store(a.agg_out + (size_t)(row0 + r) * K + col0, s);
            }
            __syncthreads();
        }
    } else {
        // rows are contiguous: element i of the tile's part of x is row i / K, column i % K
        for (int i = tid; i < R * 16; i += kBlock) {
            const int c = KP - 16 + (i & 15);
            if (c >= K || (i >> 4) >= rows) tile[(i >> 4) * LD + c] = 0.f;
        }
        const float* src = a.x + (size_t)row0 * K;
        const int total = rows * K;
        for (int base = 0; base < total; base += kFlight * kBlock) {
            float v[kFlight];
#pragma unroll
            for (int u = 0; u < kFlight; ++u) { const int i = base + tid + u * kBlock; v[u] = i < total ? src[i] : 0.f; }
#pragma unroll
            for (int u = 0; u < kFlight; ++u) {
                const int i = base + tid + u * kBlock;
                const int r = K >= 2 ? (int)__umulhi((unsigned)i, a.k_magic) : i;
                if (i < total) tile[r * LD + i - r * K] = v[u];
            }
        }
        __syncthreads();
    }

    // ---- 2. the product: lane (q, t) supplies row t's k = k0 + 4 q + s at instruction s and ends up with columns 4 q .. + 3 of
    // that row of a block
    mfma_f4 acc[NB][RT];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[b][i] = mfma_f4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < KP; k0 += 16) {
        float wn[NB][4];
        load_w(k0 + 16, wn);                                   // past the end: zeros, nothing is read
        float4 x[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) x[i] = *reinterpret_cast<const float4*>(tile + (16 * i + t) * LD + k0 + 4 * q);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (b >= nb) continue;                          // uniform
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][0], x[i].x, acc[b][i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][1], x[i].y, acc[b][i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][2], x[i].z, acc[b][i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < RT; ++i) acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][3], x[i].w, acc[b][i], 0, 0, 0);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) wf[b][s] = wn[b][s];
    }
    __syncthreads();                                           // the left operand has been read
    auto put = [&](int row_block, int col_block, const mfma_f4& v) {
        const int col = col_block + 4 * q;
        float* dst = tile + (16 * row_block + t) * n + col;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (col + j < n) dst[j] = v[j];
    };
#pragma unroll
    for (int b = 0; b < NB; ++b)
        if (b < nb) {
#pragma unroll
            for (int i = 0; i < RT; ++i) put(i, 16 * (wave + kWaves * b), acc[b][i]);
        }

    // ---- 3. flat words of the tile's rows; everything they wait for from memory is asked for at once
    constexpr int EX = R * 64 * NB / (4 * kBlock);
    const size_t flat0 = (size_t)row0 * n;
    const int total = rows * n;
    auto load = [&](const float* p, int i) {
        float4 v = f4_zero();
        if (i + 4 <= total) return V::load(p + flat0 + i);
        if (i < total) v.x = p[flat0 + i];
        if (i + 1 < total) v.y = p[flat0 + i + 1];
        if (i + 2 < total) v.z = p[flat0 + i + 2];
        return v;
    };
    auto store = [&](float* p, int i, const float4& v) {
        if (i + 4 <= total) { V::store(p + flat0 + i, v); return; }
        p[flat0 + i] = v.x;
        if (i + 1 < total) p[flat0 + i + 1] = v.y;
        if (i + 2 < total) p[flat0 + i + 2] = v.z;
    };
    const float* first = a.msg ? a.msg : a.gate;
    float4 ex[EX], ac[WT ? EX : 1];
#pragma unroll
    for (int u = 0; u < EX; ++u) ex[u] = first ? load(first, 4 * (tid + u * kBlock)) : f4_zero();
    if constexpr (WT) {
#pragma unroll
        for (int u = 0; u < EX; ++u) ac[u] = a.acc ? load(a.acc, 4 * (tid + u * kBlock)) : f4_zero();
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < EX; ++u) {
        const int i = 4 * (tid + u * kBlock);
        if (i < total) {
            float4 v = *reinterpret_cast<const float4*>(tile + i);
            if (a.bias) { v.x += a.bias[i % n]; v.y += a.bias[(i + 1) % n]; v.z += a.bias[(i + 2) % n]; v.w += a.bias[(i + 3) % n]; }
            if (a.msg) v = V::add(v, ex[u]);
            if constexpr (WT) {
                if (a.gate)
                    v = make_float4(ex[u].x > 0.f ? v.x : 0.f, ex[u].y > 0.f ? v.y : 0.f, ex[u].z > 0.f ? v.z : 0.f, ex[u].w > 0.f ? v.w : 0.f);
            }
            if (a.relu) v = relu_ref4(v);
            store(a.out, i, v);
            if (a.relu_out) store(a.relu_out, i, relu_ref4(v));
            if constexpr (WT) {
                if (a.acc) store(a.acc, i, V::add(ac[u], v));
            }
        }
    }
}

// The same for few rows, where a launch is one chain of waits and the matrix instructions of a workgroup are those of one compute unit: a
// workgroup takes 16 rows and a share of the columns, a row is summed by a lane group of its own, a wavefront has one block of 16
// columns of W, all of it in registers, and the product follows behind one barrier, straight to memory.  (W a step of 16 k ahead of the
// product, as above, is a trip to L2 per step where nothing else runs.)  The workgroups that share a product sum its rows each; the
// sums have the order of the kernel above.  286 rows, hidden 252: 19.3 -> 6.7 us per level; hidden 100 8.3 -> 5.7, 50 5.3 -> 4.6; 1,760
// rows, hidden 200 16.7 -> 7.6, backward 16.3 -> 9.1.
// BLOCKS: wavefronts, blocks of 16 columns that the left operand has at most.
template <int BLOCKS, bool GATHER, bool WT>
__global__ __launch_bounds__(BLOCKS * kWave) void s2v_rows_few_kernel(RowsArgs a, int blocks)
{
    using V = ColsLoose;
    constexpr int kThreads = BLOCKS * kWave;
    constexpr int FL = BLOCKS == 16 ? 4 : kFlight;             // W takes 64 of 128 registers there
    extern __shared__ float4 smem4[];
    __shared__ float4 shared4[GATHER ? kBlock : 1];            // sums of a long row
    __shared__ int long_row[GATHER ? 16 : 1];
    __shared__ int long_count;
    float* tile = reinterpret_cast<float*>(smem4);             // [16][LD]
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int K = a.K, n = a.n;
    const int KP = (K + 15) & ~15, LD = KP + 4;
    const long long row0 = (long long)blockIdx.x * 16;
    const int rows = (int)min(16ll, (long long)a.N - row0);

    const int units = (K + 3) / 4;
    const int logG = units <= 1 ? 0 : 32 - __builtin_clz((unsigned)(units - 1));
    const int G = 1 << logG, sub = tid & (G - 1), grp = tid >> logG;      // at least 16 groups
    const bool live = sub < units;
    const int col0 = V::at(sub, K);
    // blocks: of the product, per workgroup; the workgroups of a row of the grid's y share the 16 rows' product
    const int block = blockIdx.y * blocks + wave;
    const bool wave_live = wave < blocks && 16 * block < n;    // uniform

    float wf[BLOCKS][4];                                       // wf[k][s] = W[16 k + 4 q + s][16 block + t], zero from k = K on
    auto ask_w = [&]() {
        const rsrc_t w_rsrc = make_rsrc(a.W, (unsigned)((size_t)K * n * 4));
        const int w_col = 16 * block + t;
#pragma unroll
        for (int k = 0; k < BLOCKS; ++k) {
            if (16 * k >= KP || !wave_live) { wf[k][0] = wf[k][1] = wf[k][2] = wf[k][3] = 0.f; continue; }     // uniform
            if constexpr (WT) {
                if (16 * k + 16 <= K) {
                    const float4 w = V::load(a.W + (size_t)min(w_col, n - 1) * K + 16 * k + 4 * q);
                    wf[k][0] = w.x; wf[k][1] = w.y; wf[k][2] = w.z; wf[k][3] = w.w;
                    continue;
                }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int at = 16 * k + 4 * q + s;
                wf[k][s] = buf_load_f(w_rsrc, at < K && w_col < n ? (WT ? w_col * K + at : at * n + w_col) * 4 : kBufPastEnd, 0);
            }
        }
    };
    // columns out_col .. + 3 of row t of the product are this lane's
    const int out_col = 16 * block + 4 * q;
    const size_t out_at = (size_t)(row0 + min(t, rows - 1)) * n + out_col;
    auto ask = [&](const float* p) {
        float4 v = f4_zero();
        if (!p || t >= rows || !wave_live) return v;
        if (out_col + 4 <= n) return V::load(p + out_at);
        if (out_col < n) v.x = p[out_at];
        if (out_col + 1 < n) v.y = p[out_at + 1];
        if (out_col + 2 < n) v.z = p[out_at + 2];
        return v;
    };
    float4 ex = f4_zero(), old = f4_zero();
    auto ask_rest = [&]() {                                    // what the product is multiplied with and what is added to it
        ask_w();
        ex = ask(a.msg ? a.msg : a.gate);
        if constexpr (WT) old = ask(a.acc);
    };

    // ---- the left operand's rows
    if constexpr (GATHER) {
        // Row pointers, entries, rows: three trips to memory, one after the other (buffer loads: what there is not is asked for past
        // the end).  The rest is asked for behind the first rows and arrives with them.
        int start = 0, end = 0;
        {
            const rsrc_t rp_rsrc = make_rsrc(a.row_ptr, (unsigned)(a.N + 1) * 4u);
            start = buf_load_i(rp_rsrc, grp < rows ? (int)(row0 + grp) * 4 : kBufPastEnd, 0);
            end = buf_load_i(rp_rsrc, grp < rows ? (int)(row0 + grp + 1) * 4 : kBufPastEnd, 0);
        }
        if (tid == 0) long_count = 0;
        for (int i = tid; i < 16 * 16; i += kThreads) {        // the columns behind K
            const int c = KP - 16 + (i & 15);
            if (c >= K) tile[(i >> 4) * LD + c] = 0.f;
        }
        const rsrc_t col_rsrc = make_rsrc(a.col_idx, 0xFFFFFFFCu), val_rsrc = make_rsrc(a.val, 0xFFFFFFFCu);
        const rsrc_t x_rsrc = make_rsrc(a.x, (unsigned)a.N * (unsigned)K * 4u);
        const bool is_long = end - start > kLongRow;
        const int stop = is_long ? start : end;
        int c[FL];
        float v[FL];
        float4 x[FL];
        auto ask_entries = [&](int base) {
#pragma unroll
            for (int u = 0; u < FL; ++u) {
                const int off = base + u < stop ? (base + u) * 4 : kBufPastEnd;
                c[u] = buf_load_i(col_rsrc, off, 0);
                v[u] = buf_load_f(val_rsrc, off, 0);
            }
        };
        auto ask_rows = [&](int base) {
#pragma unroll
            for (int u = 0; u < FL; ++u) x[u] = buf_load4(x_rsrc, base + u < stop && live ? (c[u] * K + col0) * 4 : kBufPastEnd, 0);
        };
        float4 sum = f4_zero();
        auto add_rows = [&](int base, const float (&w)[FL]) {
#pragma unroll
            for (int u = 0; u < FL; ++u)
                if (base + u < stop) f4_fma(sum, w[u], a.relu_in ? relu_ref4(x[u]) : x[u]);
        };
        ask_entries(start);
        ask_rows(start);
        ask_rest();
        for (int base = start; base < stop; base += FL) {
            float now[FL];
#pragma unroll
            for (int u = 0; u < FL; ++u) now[u] = v[u];
            const bool more = base + FL < stop;
            if (more) ask_entries(base + FL);
            add_rows(base, now);
            if (more) ask_rows(base + FL);
        }
        auto finish_row = [&](int r, const float4& total) {
            if (!live) return;
            V::store(tile + r * LD + col0, total);
            if (a.agg_out && r < rows && blockIdx.y == 0) V::store(a.agg_out + (size_t)(row0 + r) * K + col0, total);
        };
        if (grp < 16 && !is_long) finish_row(grp, sum);
        __syncthreads();
        if (is_long && grp < 16 && sub == 0) long_row[atomicAdd(&long_count, 1)] = grp;
        __syncthreads();
        const int nlong = long_count;
        const int lgroups = kBlock >> logG;                    // those of the kernel above: the same sums
        for (int li = 0; li < nlong; ++li) {
            const int r = long_row[li];
            const int first = a.row_ptr[row0 + r], last = a.row_ptr[row0 + r + 1];
            float4 total = f4_zero();
            if (grp < lgroups) {
                for (int e = first + grp; e < last; e += 4 * lgroups) {
                    int lc[4];
                    float lv[4];
                    float4 lx[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const bool ok = e + u * lgroups < last;
                        lc[u] = ok ? a.col_idx[e + u * lgroups] : 0;
                        lv[u] = ok ? a.val[e + u * lgroups] : 0.f;
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) lx[u] = e + u * lgroups < last && live ? V::load(a.x + (size_t)lc[u] * K + col0) : f4_zero();
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (e + u * lgroups < last) f4_fma(total, lv[u], a.relu_in ? relu_ref4(lx[u]) : lx[u]);
                }
                shared4[tid] = total;
            }
            __syncthreads();
            if (grp == 0) {
                float4 s = f4_zero();
                for (int g = 0; g < lgroups; ++g) s = V::add(s, shared4[g * G + sub]);
                finish_row(r, s);
            }
            __syncthreads();
        }
    } else {
        ask_rest();
        for (int i = tid; i < 16 * 16; i += kThreads) {
            const int c = KP - 16 + (i & 15);
            if (c >= K || (i >> 4) >= rows) tile[(i >> 4) * LD + c] = 0.f;
        }
        const float* src = a.x + (size_t)row0 * K;
        const int total = rows * K;
        for (int base = 0; base < total; base += 4 * kThreads) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { const int i = base + tid + u * kThreads; v[u] = i < total ? src[i] : 0.f; }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = base + tid + u * kThreads;
                const int r = K >= 2 ? (int)__umulhi((unsigned)i, a.k_magic) : i;
                if (i < total) tile[r * LD + i - r * K] = v[u];
            }
        }
        __syncthreads();
    }
    if (!wave_live) return;                                   // uniform; no barrier follows

    // ---- the product, and what follows it, straight from the registers
    mfma_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < BLOCKS; ++k) {
        if (16 * k >= KP) continue;                            // uniform
        const float4 x = *reinterpret_cast<const float4*>(tile + t * LD + 16 * k + 4 * q);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[k][0], x.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[k][1], x.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[k][2], x.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[k][3], x.w, acc, 0, 0, 0);
    }
    if (t >= rows) return;
    float4 v = make_float4(acc[0], acc[1], acc[2], acc[3]);
    if (a.bias) {
        const int last = n - 1;
        v.x += a.bias[min(out_col, last)]; v.y += a.bias[min(out_col + 1, last)]; v.z += a.bias[min(out_col + 2, last)]; v.w += a.bias[min(out_col + 3, last)];
    }
    if (a.msg) v = V::add(v, ex);
    if constexpr (WT) {
        if (a.gate) v = make_float4(ex.x > 0.f ? v.x : 0.f, ex.y > 0.f ? v.y : 0.f, ex.z > 0.f ? v.z : 0.f, ex.w > 0.f ? v.w : 0.f);
    }
    if (a.relu) v = relu_ref4(v);
    auto put = [&](float* p, const float4& x) {
        if (out_col + 4 <= n) { V::store(p + out_at, x); return; }
        if (out_col < n) p[out_at] = x.x;
        if (out_col + 1 < n) p[out_at + 1] = x.y;
        if (out_col + 2 < n) p[out_at + 2] = x.z;
    };
    put(a.out, v);
    if (a.relu_out) put(a.relu_out, relu_ref4(v));
    if constexpr (WT) {
        if (a.acc) put(a.acc, V::add(old, v));
    }
}

template <int BLOCKS, bool GATHER, bool WT>
int launch_rows_few(const RowsArgs& a, hipStream_t s)
{
    const int KP = (a.K + 15) & ~15;
    const int tiles = (int)(((long long)a.N + 15) / 16), blocks = (a.n + 15) / 16;
    // as long as there are compute units for it, four blocks to a workgroup: the matrix instructions of 16 x 256 x 256 on one of them take 4 us
    // (in place, rows are read by nobody else: the input stage with as many feature columns as hidden units)
    int share = a.x == a.out || a.x == a.relu_out ? 1 : (blocks + 3) / 4;
    while (share > 1 && share * tiles > kNumCU) --share;
    const int per = (blocks + share - 1) / share;
    hipLaunchKernelGGL((s2v_rows_few_kernel<BLOCKS, GATHER, WT>), dim3(tiles, share), dim3(BLOCKS * kWave), sizeof(float) * 16 * (KP + 4), s, a, per);
    GNNHIP_LAUNCH_CHECK("s2v_rows_few");
    return GNNHIP_OK;
}

template <int RT, int NB, int MINW, bool GATHER, bool WT>
int launch_rows(const RowsArgs& a, hipStream_t s)
{
    const int KP = (a.K + 15) & ~15;
    const int width = KP + 4 > a.n ? KP + 4 : a.n;
    const unsigned grid = (unsigned)(((long long)a.N + 16 * RT - 1) / (16 * RT));
    constexpr bool kGated = !WT && NB <= 2;                // input and levels of batch_forward.hip's sizes
    if (!kGated && a.launch_gate) return GNNHIP_EUNSUPPORTED;
    const auto kernel = kGated && a.launch_gate ? &s2v_rows_kernel<RT, NB, MINW, GATHER, WT, kGated> : &s2v_rows_kernel<RT, NB, MINW, GATHER, WT, false>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), sizeof(float) * 16 * RT * width, s, a);
    GNNHIP_LAUNCH_CHECK("s2v_rows");
    return GNNHIP_OK;
}

// Rows per tile for products of up to 128 columns.  Few rows: 16, so that there is a workgroup for every compute unit.  Many: 64, which
// use every fetched word of W four times.  In between the tiles of 64 rows leave each compute unit one or two workgroups,
// whose phases have nothing to hide behind, and 32 rows are the better ones (hidden 85, 22,000 nodes: 21.0 -> 15.4 us per
// level, 24.7 -> 18.3 backward; 38,000: 29.7 -> 24.5), up to the 49,152 rows that six workgroups per compute unit hold at once
// where the registers allow so many (from 40,960 on: 48,750 nodes, hidden 36 to 100 6 to 12 % less; below, the registers
// that this takes away cost 3 %; up to 8 columns a tile is one short phase, and 64 rows are the faster ones there: hidden 4, 45,000
// nodes 9.9 us, 10.4 with 32 rows; hidden 125 to 127 backward lose 1 to 4 % from 43,000 nodes on with 2.2 entries per row and gain 2 to 3 with 8).
// 51,000 nodes take two rounds: 2 to 8 % slower than 64 rows.
template <int NB, bool GATHER, bool WT>
int rows_by_tile(const RowsArgs& a, hipStream_t s)
{
    if (a.N < 64 * kNumCU) return launch_rows<1, NB, 3, GATHER, WT>(a, s);
    if (a.N < 160 * kNumCU) return launch_rows<2, NB, 3, GATHER, WT>(a, s);
    if (a.N <= 6 * 32 * kNumCU && a.n > 8) return launch_rows<2, NB, 6, GATHER, WT>(a, s);
    return launch_rows<4, NB, 3, GATHER, WT>(a, s);
}

// nnz: entries of A (GATHER)
template <bool GATHER, bool WT>
int rows_dispatch(RowsArgs a, long long nnz, hipStream_t s)
{
    a.k_magic = a.K >= 2 ? (unsigned)(((1ull << 32) + a.K - 1) / a.K) : 0;
    // A workgroup per 16 rows: a second one per compute unit would wait for the first (4,112 rows, hidden 200, backward 18.8 -> 20.5 us).  Up to 64
    // columns nothing is shared out, and all that is gained is W's way into registers beside the first rows: rows of many entries, and of more
    // than columns, are summed faster in the kernel of many rows (2,048 rows, level and backward, there and here: hidden 20, 5 entries per row 4.3 us and 4.0,
    // 4.7 and 4.4; 16 5.0 and 4.9, 5.5 and 5.3; 30 6.4 and 6.6, 6.8 and 7.0; 60 9.2 and 10.4, 9.7 and 10.7; hidden 50, 16 5.6 and 5.2, 60 9.8 and
    // 11.1; hidden 8, 5 4.2 and 4.0; 12 4.9 and 4.8, 5.2 and 5.3; 30 6.6 and 6.9, 6.9 and 7.5; 180 24.5 and 27.4, 24.7 and 28.3)
    const int widest = a.K > a.n ? a.K : a.n;
    const bool many_entries = GATHER && widest <= 64 && nnz > (a.K < 16 ? a.K : 16) * (long long)a.N;
    if (a.N <= kFewRows && a.K >= 4 && !many_entries && !a.launch_gate) {          // (these have no gated variants)
        if (widest <= 64) return launch_rows_few<4, GATHER, WT>(a, s);
        if (widest <= 128) return launch_rows_few<8, GATHER, WT>(a, s);
        return launch_rows_few<16, GATHER, WT>(a, s);
    }
    if (a.n <= 64) return rows_by_tile<1, GATHER, WT>(a, s);
    if (a.n <= 128) return rows_by_tile<2, GATHER, WT>(a, s);
    // wider: 32 rows, where the tile leaves room for two workgroups per compute unit
    return a.N < 64 * kNumCU ? launch_rows<1, 4, 3, GATHER, WT>(a, s) : launch_rows<2, 4, 3, GATHER, WT>(a, s);
}

}  // namespace

namespace {
// Whether the gathered products below take a matrix of this size.  Denser ones go through the SpMM, which cuts long rows into
// pieces from kHubMinRows rows and 12 entries per row on and gives a row a workgroup from 256 entries per row on, and
// level_rows_dense_dispatch.
bool level_rows_covers(int N, int C, long long nnz)
{
    const long long mean = N >= kHubMinRows ? 12 : 256;
    return C >= 4 && C <= kMaxWidth && nnz < mean * (long long)N;
}
}  // namespace

int level_rows_dispatch(int N, int C, long long nnz, const int* row_ptr, const int* col_idx, const float* val, const float* h_in,
                        const float* W, const float* msg, const float* bias, float* h_out, bool same_graph, bool relu_in, CsrPlan* plan,
                        hipStream_t s, const int* gate)
{
    if (!level_rows_covers(N, C, nnz)) return GNNHIP_EUNSUPPORTED;
    RowsArgs a{};
    if (int rc = hub_prepass(N, C, nnz, row_ptr, col_idx, val, h_in, C, s, &a.hubs, same_graph, relu_in, kHubThreshold, kHubChunk, -1,
                             plan ? &plan->row_hub : nullptr, gate))
        return rc;
    a.N = N; a.K = C; a.n = C;
    a.row_ptr = row_ptr; a.col_idx = col_idx; a.val = val; a.x = h_in; a.W = W;
    a.bias = bias; a.msg = msg; a.out = h_out; a.relu = 1; a.relu_in = relu_in; a.launch_gate = gate;
    return rows_dispatch<true, false>(a, nnz, s);
}

int level_rows_backward_dispatch(int N, int C, long long nnz, const int* row_ptr, const int* col_idx, const float* val, const float* dz,
                                 const float* W, float* u, float* g_prev, const float* gate, float* acc, hipStream_t s)
{
    if (!level_rows_covers(N, C, nnz)) return GNNHIP_EUNSUPPORTED;
    RowsArgs a{};
    if (int rc = hub_prepass(N, C, nnz, row_ptr, col_idx, val, dz, C, s, &a.hubs)) return rc;
    a.N = N; a.K = C; a.n = C;
    a.row_ptr = row_ptr; a.col_idx = col_idx; a.val = val; a.x = dz; a.W = W;
    a.gate = gate; a.agg_out = u; a.out = g_prev; a.acc = acc;
    return rows_dispatch<true, true>(a, nnz, s);
}

// out = x * W (+ bias + msg); relu: out = ReLU of that; relu_out (or null) = ReLU(out).  x [N, K], W [K, n].
int level_rows_dense_dispatch(int N, int K, int n, const float* x, const float* W, const float* bias, const float* msg, float* out,
                              bool relu, float* relu_out, hipStream_t s, const int* gate)
{
    // (64 rows of more than 252 columns would not fit 64 KB of LDS)
    if (K < 1 || K > (n <= 128 ? 128 : kMaxWidth) || n > kMaxWidth) return GNNHIP_EUNSUPPORTED;
    RowsArgs a{};
    a.N = N; a.K = K; a.n = n;
    a.x = x; a.W = W; a.bias = bias; a.msg = msg; a.out = out; a.relu = relu; a.relu_out = relu_out; a.launch_gate = gate;
    return rows_dispatch<false, false>(a, 0, s);
}

}  // namespace gnnhip
