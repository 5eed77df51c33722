// Balanced pre-pass for high-degree rows ("hubs") of a CSR matrix.
//
// The SpMM and fused-level kernels give a row to a group of lanes, which is right
// for the short rows of molecule batches and of uniform random graphs but leaves
// one group, or one workgroup, alone with a row of 10^5 entries on a power-law
// graph (R-MAT, a = 0.57: the largest of 4M rows holds 160,000 of 64M entries, and
// the hubs sit next to each other at the low row indices).  Rows with more than
// kHubThreshold entries are therefore summed here, ahead of the consumer kernel,
// with the work cut by entries instead of by rows:
//
//   count   per run of rows: its hubs and how many chunks (kHubChunk entries each) they have
//   partial one wavefront per chunk: it finds its chunk's row from the counts, which every workgroup adds up, and the
//           run's hubs, sums val * B[col, :] over the chunk, and the wavefront of a hub's first chunk leaves the number
//           of that chunk in row_chunk[row] (written for hubs only)
//
// The consumer takes a row whose length exceeds the threshold from the sums of its chunks, row_chunk[row] and the
// following ones, added in chunk order (hub_row_sum).  Every sum is taken in an order fixed by the matrix structure,
// so the result does not depend on scheduling: no atomics, no communication inside a launch.
//
// Most matrices have no hubs, and then the pass is nothing but its launches: with a launch that turned the counts into
// one list of all chunks and a launch that added up the chunks of a hub it was four per product instead of two.
#include "columns.h"
#include "graph_bins.h"

#include <map>

namespace gnnhip {

namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kRunRows = 1024;               // four rows per lane of the counting workgroup
constexpr int kMaxRuns = 1024;               // counts per matrix: runs get longer past 1M rows

__device__ __forceinline__ int hub_chunks(int deg, int threshold, int shift) { return deg > threshold ? (deg + (1 << shift) - 1) >> shift : 0; }

__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(v, d, kWave);
        if (lane >= d) v += o;
    }
    return v;
}

// The last of n ascending values that is no more than x (the first one is); by a wavefront, 64 samples a step.
__device__ __forceinline__ int last_at_most(const int* v, int n, int x)
{
    const int lane = threadIdx.x & (kWave - 1);
    int base = 0;
    for (;;) {
        const int step = (n + kWave - 1) / kWave;
        const unsigned long long a = __ballot(lane * step < n && v[base + min(lane * step, n - 1)] <= x);
        const int at = (63 - __clzll((long long)a)) * step;
        base += at;
        if (step == 1) return base;
        n = min(step, n - at);
    }
}

// One run of `rows` rows, by a workgroup: its hubs in row order (list_row) with the chunks of the run ahead of each
// (list_chunk), both from the run's first row on, and the numbers of its hubs and of their chunks.
__device__ __forceinline__ void count_run(int run, int m, int rows, const int* __restrict__ row_ptr, int* __restrict__ run_hubs,
                                          int* __restrict__ run_chunks, int* __restrict__ list_row, int* __restrict__ list_chunk, int threshold, int shift)
{
    __shared__ int sh[2][kWavesPerBlock];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const long long lo = (long long)run * rows, hi = min(lo + rows, (long long)m);
    int hubs = 0, chunks = 0;                    // of the rows before the ones in hand
    for (long long base = lo; base < hi; base += kBlock * 4) {
        const long long r0 = base + threadIdx.x * 4;
        int p[5], h = 0, c = 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) p[i] = row_ptr[min(r0 + i, hi)];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int nc = hub_chunks(p[i + 1] - p[i], threshold, shift);
            h += nc > 0;
            c += nc;
        }
        if (!__syncthreads_or(h)) continue;      // most runs of most matrices
        const int ih = wave_inclusive_scan(h), ic = wave_inclusive_scan(c);
        if (lane == kWave - 1) { sh[0][wave] = ih; sh[1][wave] = ic; }
        __syncthreads();
        int at_h = hubs + ih - h, at_c = chunks + ic - c;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) {
            if (w < wave) { at_h += sh[0][w]; at_c += sh[1][w]; }
            hubs += sh[0][w];
            chunks += sh[1][w];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int nc = hub_chunks(p[i + 1] - p[i], threshold, shift);
            if (nc > 0) {
                list_row[lo + at_h] = (int)(r0 + i);
                list_chunk[lo + at_h] = at_c;
                ++at_h;
                at_c += nc;
            }
        }
        __syncthreads();                         // sh is rewritten by the next rows
    }
    if (threadIdx.x == 0) { run_hubs[run] = hubs; run_chunks[run] = chunks; }
}

__global__ __launch_bounds__(kBlock) void hub_count_kernel(int m, int rows, const int* __restrict__ row_ptr, int* __restrict__ run_hubs,
                                                           int* __restrict__ run_chunks, int* __restrict__ list_row,
                                                           int* __restrict__ list_chunk, int threshold, int shift)
{
    count_run((int)blockIdx.x, m, rows, row_ptr, run_hubs, run_chunks, list_row, list_chunk, threshold, shift);
}

// The same and, by the workgroups behind, the bins of a batch that may be one of small graphs (graph_bins.h): neither waits for the other, and a
// launch of its own costs either about as long as both take together (44,643 nodes in 1,500 graphs: 4.8 us and 4.0 in a trace).
__global__ __launch_bounds__(kBlock) void hub_count_bins_kernel(int runs, int m, int rows, const int* __restrict__ row_ptr, int* __restrict__ run_hubs,
                                                                int* __restrict__ run_chunks, int* __restrict__ list_row,
                                                                int* __restrict__ list_chunk, int threshold, int shift, BinsArgs bins)
{
    if ((int)blockIdx.x < runs) {
        count_run((int)blockIdx.x, m, rows, row_ptr, run_hubs, run_chunks, list_row, list_chunk, threshold, shift);
    } else {
        pack_segment<true>(__builtin_amdgcn_readfirstlane((int)(((int)blockIdx.x - runs) * kWavesPerBlock + threadIdx.x / kWave)), bins);
    }
}

// One wavefront per chunk.  The wavefront is split into 64 / G lane groups; group g takes the
// chunk's entries g, g + ngroups, ... eight at a time, a lane owns the column slabs
// (sub + it * G) * V::kVec.  The groups' sums are added through LDS in group order.
template <class V, int ITERS, bool GATED>
__global__ __launch_bounds__(kBlock) void hub_partial_kernel(
    int run_rows, int runs, const int* __restrict__ run_hubs, const int* __restrict__ run_chunks, const int* __restrict__ list_row,
    const int* __restrict__ list_chunk, int chunk_cap, int n, const int* __restrict__ row_ptr, const int* __restrict__ col_idx, const float* __restrict__ val, const float* __restrict__ B, int ldb, int logG,
    int* __restrict__ row_chunk, float* __restrict__ part, int ldp, int relu_in, int threshold, int shift, const int* __restrict__ gate)
{
    // relu_in: the rows of B are used as ReLU(B) (a first level that reads msg in place of h0)
    __shared__ float red[kWavesPerBlock][kWave * V::kVec * ITERS];
    __shared__ int before[kMaxRuns + 1];         // chunks ahead of a run
    __shared__ int wave_total[kWavesPerBlock];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int G = 1 << logG, sub = lane & (G - 1), grp = lane >> logG, ngroups = kWave >> logG;
    const int width = G * V::kVec * ITERS;

    int nchunks;
    {
        constexpr int kEach = kMaxRuns / kBlock;
        const int per = (runs + kBlock - 1) / kBlock;            // consecutive counts of a lane, kEach at most
        int v[kEach], mine = 0;
#pragma unroll
        for (int i = 0; i < kEach; ++i) v[i] = i < per && threadIdx.x * per + i < runs ? run_chunks[threadIdx.x * per + i] : 0;
#pragma unroll
        for (int i = 0; i < kEach; ++i) mine += v[i];
        const int incl = wave_inclusive_scan(mine);
        if (lane == kWave - 1) wave_total[wave] = incl;
        __syncthreads();
        int at = incl - mine;
        nchunks = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) {
            if (w < wave) at += wave_total[w];
            nchunks += wave_total[w];
        }
        if (nchunks == 0) return;
        // (here and not ahead of the counts: most matrices have no long rows, and the word would be a trip to memory of its own)
        if (gated_off<GATED>(gate)) return;
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            if (i < per && threadIdx.x * per + i < runs) before[threadIdx.x * per + i] = at;
            at += v[i];
        }
        __syncthreads();
    }

    for (int c = blockIdx.x * kWavesPerBlock + wave; c < nchunks; c += gridDim.x * kWavesPerBlock) {
        // the run that holds chunk c, and in it the hub
        const int run = last_at_most(before, runs, c), rest = c - before[run];
        const int* first_chunk = list_chunk + (size_t)run * run_rows;
        const int at = last_at_most(first_chunk, run_hubs[run], rest);
        const int row = list_row[(size_t)run * run_rows + at], within = rest - first_chunk[at];
        const int rb = row_ptr[row], re = row_ptr[row + 1];
        // a hub past the capacity of the buffers keeps -1: its consumer sums it in place
        const bool fits = c - within + hub_chunks(re - rb, threshold, shift) <= chunk_cap;
        if (within == 0 && lane == 0) row_chunk[row] = fits ? c : -1;
        if (!fits) continue;
        const int cb = rb + (within << shift);
        const int ce = min(cb + (1 << shift), re);
        typename V::T acc[ITERS];
#pragma unroll
        for (int it = 0; it < ITERS; ++it) acc[it] = V::zero();
        // eight entries of the group at a time, the last ones of the chunk under a predicate (a serial tail would
        // walk up to seven dependent index -> row loads one after the other, and most chunks of the matrices that
        // pick partial sums are shorter than one such block); the order of the additions is the entries' order
        for (int t = cb + grp; t < ce; t += 8 * ngroups) {
            int c8[8];
            float v8[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const bool ok = t + u * ngroups < ce;
                // no index array: entry t of the row is column t with weight 1 (a matrix that picks consecutive rows of B,
                // whose row loads then wait for no index load)
                c8[u] = !ok ? 0 : col_idx ? col_idx[t + u * ngroups] : t + u * ngroups;
                v8[u] = !ok ? 0.f : val ? val[t + u * ngroups] : 1.f;
            }
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int unit = sub + it * G;
                if (unit * V::kVec < n) {
                    const int col0 = V::at(unit, n);
                    typename V::T x[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        x[u] = (t + u * ngroups < ce) ? V::load(B + (size_t)c8[u] * ldb + col0) : V::zero();
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (t + u * ngroups < ce) V::fma(acc[it], v8[u], relu_in ? V::relu(x[u]) : x[u]);
                }
            }
        }
#pragma unroll
        for (int it = 0; it < ITERS; ++it) V::store(red[wave] + grp * width + (sub + it * G) * V::kVec, acc[it]);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        float* dst = part + (size_t)c * ldp;
        if (grp == 0) {
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int unit = sub + it * G;
                if (unit * V::kVec < n) {
                    typename V::T s = V::zero();
                    for (int g = 0; g < ngroups; ++g) s = V::add(s, V::load(red[wave] + g * width + unit * V::kVec));
                    V::store(dst + V::at(unit, n), s);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");       // red[wave] is rewritten by the next chunk
    }
}

inline int ilog2_ceil_(int x)
{
    int l = 0;
    while ((1 << l) < x) ++l;
    return l;
}

inline size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

}  // namespace

namespace {

// Where the arrays of one pre-pass lie inside its block; everything up to `part` does not depend on the width n.
struct HubLayout {
    int run_rows, runs, chunk_cap, ldp;
    size_t o_hubs, o_chunks, o_lrow, o_lchunk, o_row, o_part, bytes;
};

HubLayout hub_layout(int m, int n, long long nnz, int threshold, int chunk_len, long long max_hubs)
{
    HubLayout L;
    L.ldp = (int)round_up((size_t)n, 4);
    L.run_rows = (int)round_up((size_t)(m + kMaxRuns - 1) / kMaxRuns, kRunRows);
    L.runs = (m + L.run_rows - 1) / L.run_rows;
    long long hub_cap = nnz / (threshold + 1) + 1;
    if (max_hubs >= 0 && max_hubs < hub_cap) hub_cap = max_hubs;
    L.chunk_cap = (int)(nnz / chunk_len + hub_cap + 1);
    size_t off = 0;
    auto carve = [&](size_t bytes) { const size_t o = off; off = round_up(off + bytes, 256); return o; };
    L.o_hubs = carve(sizeof(int) * L.runs);
    L.o_chunks = carve(sizeof(int) * L.runs);
    L.o_lrow = carve(sizeof(int) * (size_t)L.runs * L.run_rows);
    L.o_lchunk = carve(sizeof(int) * (size_t)L.runs * L.run_rows);
    L.o_row = carve(sizeof(int) * (size_t)m);
    L.o_part = carve(sizeof(float) * (size_t)L.chunk_cap * L.ldp);
    L.bytes = off;
    return L;
}

template <class V, int ITERS>
void launch_partial(hipStream_t s, const HubLayout& L, char* base, int n, const int* row_ptr, const int* col_idx, const float* val,
                    const float* B, int ldb, int logG, int relu_in, int threshold, int shift, const int* gate)
{
    // a wavefront per chunk the matrix can have, up to eight workgroups per compute unit
    long long grid = ((long long)L.chunk_cap + kWavesPerBlock - 1) / kWavesPerBlock;
    if (grid > kNumCU * 8) grid = kNumCU * 8;
    auto ints = [base](size_t o) { return reinterpret_cast<int*>(base + o); };
    const auto kernel = gate ? &hub_partial_kernel<V, ITERS, true> : &hub_partial_kernel<V, ITERS, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, L.run_rows, L.runs, ints(L.o_hubs),
                       ints(L.o_chunks), ints(L.o_lrow), ints(L.o_lchunk), L.chunk_cap, n, row_ptr, col_idx, val, B, ldb, logG,
                       ints(L.o_row), reinterpret_cast<float*>(base + L.o_part), L.ldp, relu_in, threshold, shift, gate);
}

inline bool hub_pass_applies(int m, int n, long long nnz, int threshold) { return !(m < kHubMinRows || nnz <= threshold || n > kWave * 16); }

// What the stream's scratch slot holds a plan for.  Kept per stream, next to the scratch it describes (any thread
// that plans on the stream replaces it), not per thread.
struct HubMemo {
    const int* row_ptr;
    int m, n;
    long long nnz;
    void* base;
    int threshold, chunk_len, chunk_cap;
    bool operator==(const HubMemo& o) const
    {
        return row_ptr == o.row_ptr && m == o.m && n == o.n && nnz == o.nnz && base == o.base && threshold == o.threshold && chunk_len == o.chunk_len &&
               chunk_cap == o.chunk_cap;
    }
};

// Whether the stream's scratch slot holds this plan already, which is looked at only with `reuse`; else it is noted that it will.
bool plan_in_place(hipStream_t s, const HubMemo& memo, bool reuse)
{
    static std::mutex memo_mu;
    static std::map<hipStream_t, HubMemo> memos;
    std::lock_guard<std::mutex> lock(memo_mu);
    auto it = memos.find(s);
    if (reuse && it != memos.end() && it->second == memo) return true;
    memos[s] = memo;
    return false;
}

inline int chunk_shift(int chunk_len)
{
    int shift = 0;
    while ((1 << shift) < chunk_len) ++shift;
    return shift;
}

}  // namespace

// The bins of a batch that may be one of small graphs and, in the same launch, the counting that the levels of hidden size n over its A would begin
// with; *counted: their first hub_prepass may have reuse_plan.
int hub_count_with_bins(int m, int n, long long nnz, const int* row_ptr, const BinsArgs& bins, hipStream_t s, bool* counted)
{
    constexpr int threshold = kHubThreshold, chunk_len = kHubChunk;
    *counted = hub_pass_applies(m, n, nnz, threshold);
    if (!*counted) {
        hipLaunchKernelGGL((graph_bins_kernel<true>), dim3(ceil_div_u((size_t)bins.B, kBinBlock)), dim3(kBinBlock), 0, s, bins);
        GNNHIP_LAUNCH_CHECK("graph_bins");
        return GNNHIP_OK;
    }
    const HubLayout L = hub_layout(m, n, nnz, threshold, chunk_len, -1);
    void* base = nullptr;
    if (int rc = stream_scratch_slot(s, 1, L.bytes, &base)) return rc;
    (void)plan_in_place(s, HubMemo{row_ptr, m, n, nnz, base, threshold, chunk_len, L.chunk_cap}, false);
    char* b = static_cast<char*>(base);
    hipLaunchKernelGGL(hub_count_bins_kernel, dim3((unsigned)L.runs + ceil_div_u((size_t)bins.B, kBlock)), dim3(kBlock), 0, s, L.runs, m, L.run_rows, row_ptr,
                       reinterpret_cast<int*>(b + L.o_hubs), reinterpret_cast<int*>(b + L.o_chunks), reinterpret_cast<int*>(b + L.o_lrow),
                       reinterpret_cast<int*>(b + L.o_lchunk), threshold, chunk_shift(chunk_len), bins);
    GNNHIP_LAUNCH_CHECK("hub_count_bins");
    return GNNHIP_OK;
}

// Bytes of scratch a hub_prepass call with these arguments takes (0: the pass does not run).  A caller that must not
// fail for lack of memory after its own first launch reserves them up front (stream_scratch_slot(s, 1, ...)).
size_t hub_scratch_bytes(int m, int n, long long nnz, int threshold, int chunk_len, long long max_hubs)
{
    if (!hub_pass_applies(m, n, nnz, threshold)) return 0;
    return hub_layout(m, n, nnz, threshold, chunk_len, max_hubs).bytes;
}

// Sums the hubs of A (rows longer than `threshold` entries, cut into chunks of `chunk_len`) times B[:, 0..n) into
// plan->part.  chunk_len is a power of two.  col_idx == nullptr: entry t is column t; val == nullptr: every weight is 1.  max_hubs, when not negative, is the caller's bound on the number of such rows (it sizes the buffers).
// n <= 1024.  Without `store` the buffers live in the stream's scratch slot 1 and stay valid until the next
// hub_prepass on the same stream; with it they live in a block the store's owner keeps (pool memory, grown when a
// wider operand needs it), and the counting launch runs only while store->planned is false.
// reuse_plan (no store): the caller guarantees that the structure of A has not changed since the previous call on
// this stream with the same arguments (the levels of one forward); the counting launch is then skipped.
int hub_prepass(int m, int n, long long nnz, const int* row_ptr, const int* col_idx, const float* val,
                const float* B, int ldb, hipStream_t s, HubPlan* plan, bool reuse_plan, bool relu_in, int threshold, int chunk_len,
                long long max_hubs, HubStore* store, const int* gate)
{
    *plan = HubPlan{};
    if (!hub_pass_applies(m, n, nnz, threshold)) return GNNHIP_OK;
    const bool vec4 = (n % 4 == 0) && (ldb % 4 == 0) && aligned16(B);
    const int units = n < 4 ? n : (n + 3) / 4;
    const int logG = ilog2_ceil_(units < kWave ? units : kWave);
    const int G = 1 << logG;
    const int iters = (units + G - 1) / G;                   // 1..4
    const HubLayout L = hub_layout(m, n, nnz, threshold, chunk_len, max_hubs);
    const int shift = chunk_shift(chunk_len);

    void* base = nullptr;
    bool planned;
    if (store) {
        if (store->bytes < L.bytes) {
            if (store->base) {
                GNNHIP_HIP(hipStreamSynchronize(s));             // earlier launches may still read the old block
                (void)pool_free(store->base);
                store->base = nullptr;
                store->bytes = 0;
            }
            if (int rc = pool_acquire_exact(&store->base, L.bytes)) return rc;
            store->bytes = L.bytes;
            store->planned = false;
        }
        base = store->base;
        planned = store->planned;
        store->planned = true;
    } else {
        if (int rc = stream_scratch_slot(s, 1, L.bytes, &base)) return rc;
        planned = plan_in_place(s, HubMemo{row_ptr, m, n, nnz, base, threshold, chunk_len, L.chunk_cap}, reuse_plan);
    }
    char* b = static_cast<char*>(base);
    if (!planned) {
        hipLaunchKernelGGL(hub_count_kernel, dim3((unsigned)L.runs), dim3(kBlock), 0, s, m, L.run_rows, row_ptr,
                           reinterpret_cast<int*>(b + L.o_hubs), reinterpret_cast<int*>(b + L.o_chunks), reinterpret_cast<int*>(b + L.o_lrow),
                           reinterpret_cast<int*>(b + L.o_lchunk), threshold, shift);
    }
    if (n < 4) {
        launch_partial<ColsOne, 1>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
    } else if (vec4) {
        if (iters <= 1) launch_partial<ColsWide, 1>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
        else if (iters == 2) launch_partial<ColsWide, 2>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
        else launch_partial<ColsWide, 4>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
    } else {
        if (iters <= 1) launch_partial<ColsLoose, 1>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
        else if (iters == 2) launch_partial<ColsLoose, 2>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
        else launch_partial<ColsLoose, 4>(s, L, b, n, row_ptr, col_idx, val, B, ldb, logG, relu_in ? 1 : 0, threshold, shift, gate);
    }
    GNNHIP_LAUNCH_CHECK("hub_prepass");
    *plan = HubPlan{reinterpret_cast<int*>(b + L.o_row), reinterpret_cast<float*>(b + L.o_part), L.ldp, shift};
    return GNNHIP_OK;
}

}  // namespace gnnhip
