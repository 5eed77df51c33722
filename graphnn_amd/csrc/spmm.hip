// CSR SpMM for gfx950:  C[m,n] = alpha * A * B + beta * C,  A CSR (int32), B/C fp32 row-major.
//
// Work decomposition ("row group"): a power-of-two group of G lanes owns one CSR
// row; lane s of the group owns columns 4s..4s+3 (one 128-bit load per gathered
// row).  With n = 64 that is 16 lanes per row and 4 rows per wavefront, with
// n = 128 two rows per wavefront, with n >= 256 one row per wavefront and up to
// four column slabs per lane.  A group reads its row's column indices and values
// once, coalesced, G at a time, and hands them round with an in-group shuffle, so
// index traffic is one pass over the CSR arrays instead of one per output column.
// Gathers are issued four at a time before they are consumed to keep several
// HBM/L2 requests in flight per lane.  Accumulation is in registers in CSR order
// (deterministic, no atomics) and each output element is written exactly once.
//
// Long rows: on matrices of at least kHubMinRows rows a pre-pass (hub.hip) sums the
// rows longer than kHubThreshold entries with the work cut by entries, and the row's
// group here only scales and stores that sum.  Elsewhere rows longer than kLongRow
// entries are set aside inside the workgroup and then processed by all of its 256
// lanes together, which split the row's entries and combine the partial sums in LDS
// in a fixed order (still deterministic).
//
// Bound: HBM.  Algorithmic bytes per launch: 4(m+1) + 8 nnz + 4 k n + 4 m n.
#include "columns.h"

namespace gnnhip {
namespace {

constexpr int kBlock = 256;
constexpr int kLongRow = 2048;      // entries; longer rows are processed by the whole workgroup
constexpr long long kOneRowMeanEntries = 256;   // mean entries per row from which every row gets a workgroup (matrices below kHubMinRows rows)

// Workgroups are dealt round-robin to the 8 XCDs; give each XCD one contiguous
// slice of the row space so rows that share neighbours share an L2.
__device__ __forceinline__ unsigned xcd_remap(unsigned bid, unsigned nblocks)
{
    const unsigned per = nblocks / kNumXCD;
    const unsigned covered = per * kNumXCD;
    if (bid >= covered) return bid;
    return (bid % kNumXCD) * per + bid / kNumXCD;
}

// One row per group of G = 1 << logG lanes.  A lane owns column slabs
// (sub + it * G) * V::kVec, it < ITERS; slabs at or beyond n are skipped.
// Rows longer than long_row entries are parked in an LDS list and processed
// afterwards by the whole workgroup: group g takes entries g, g + ngroups, ...
// and the partial sums are added through LDS in group order.
// long_row < 0: one row per workgroup, summed that way whatever its length (few, long rows: pooling 1,024 nodes
// into each of 4,096 subgraphs ran one workgroup per compute unit with a lane group per row: 0.265 ms).
// RELU_IN: the rows of B count as ReLU(B).
// NARROW (G <= kNarrowGroup): a group that read its entries G at a time would have G gathers in flight, and its wavefront
// would touch a line per row and read.  The rows of a wavefront are consecutive and so are their entries: the wavefront
// copies them to LDS, coalesced, when there are at most kStaged (else every lane reads its row's entries itself), and the
// groups take eight at a time.  Sums are added in the same order.  (300,000 rows of 10 entries: width 4 77 -> 30 us, width 16
// 66 -> 55; groups of eight lanes gain 4 % there and lose 8 % at two entries per row, so the line is at four.)
constexpr int kNarrowGroup = 4;
constexpr int kStaged = 768;
template <class V, int ITERS, bool RELU_IN, bool NARROW>
__global__ __launch_bounds__(kBlock) void spmm_rowgroup_kernel(
    int m, int n, float alpha, const int* __restrict__ row_ptr, const int* __restrict__ col_idx,
    const float* __restrict__ val, const float* __restrict__ B, int ldb, float beta, float* C, int ldc,
    int logG, int long_row, HubPlan hubs)
{
    __shared__ int lr_list[kBlock];
    __shared__ int lr_count;
    __shared__ float red[kBlock * V::kVec * ITERS];      // [ngroups][G * V::kVec * ITERS]

    const int G = 1 << logG;
    const int sub = threadIdx.x & (G - 1);
    const int grp = threadIdx.x >> logG;
    const int ngroups = kBlock >> logG;
    const unsigned bid = xcd_remap(blockIdx.x, gridDim.x);
    const bool one_row = long_row < 0;
    const bool owner = !one_row || grp == 0;          // the lane group that answers for `row`
    const long long row = one_row ? (long long)bid : (long long)bid * ngroups + grp;

    if (threadIdx.x == 0) lr_count = 0;
    __syncthreads();

    int start = 0, end = 0;
    if (row < m && owner) { start = row_ptr[row]; end = row_ptr[row + 1]; }
    // a row summed by the hub pre-pass only scales and stores
    int hub = -1;
    const int entries = end - start;
    if (hubs.row_chunk && entries > kHubThreshold) hub = hubs.row_chunk[row];
    if (hub >= 0) end = start;
    const bool deferred = one_row ? (end > start) : (end - start > long_row);
    if (deferred) {
        if (sub == 0) lr_list[atomicAdd(&lr_count, 1)] = (int)row;
        end = start;      // the group idles through the main phase
    }

    typename V::T acc[ITERS];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) acc[it] = V::zero();

    if constexpr (NARROW) {
        __shared__ int2 staged[kBlock / kWave][kStaged];
        int2* mine = staged[threadIdx.x / kWave];
        const int lane = threadIdx.x & (kWave - 1);
        const int col0 = V::at(sub, n);
        constexpr int kFlight = 8;
        auto add_row = [&](auto entry) {
            for (int base = start; base < end; base += kFlight) {
                int2 cv[kFlight];
                typename V::T x[kFlight];
#pragma unroll
                for (int u = 0; u < kFlight; ++u) cv[u] = base + u < end ? entry(base + u) : make_int2(0, 0);
#pragma unroll
                for (int u = 0; u < kFlight; ++u)
                    x[u] = base + u < end && sub * V::kVec < n ? V::load(B + (size_t)cv[u].x * ldb + col0) : V::zero();
#pragma unroll
                for (int u = 0; u < kFlight; ++u)
                    if (base + u < end) V::fma(acc[0], alpha * __int_as_float(cv[u].y), RELU_IN ? V::relu(x[u]) : x[u]);
            }
        };
        // rows past the end, hubs and deferred rows are empty here and take no part in the range
        const unsigned long long busy = __ballot(end > start);
        int lo = 0, hi = 0;
        if (busy) {
            lo = __builtin_amdgcn_readlane(start, (int)__builtin_ctzll(busy));
            hi = __builtin_amdgcn_readlane(end, 63 - (int)__builtin_clzll(busy));
        }
        if (hi - lo <= kStaged) {
            for (int e = lo + lane; e < hi; e += kWave) mine[e - lo] = make_int2(col_idx[e], __float_as_int(val[e]));
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            add_row([&](int e) { return mine[e - lo]; });
        } else {
            add_row([&](int e) { return make_int2(col_idx[e], __float_as_int(val[e])); });
        }
        end = start;
    }
    for (int base = start; !NARROW && base < end; base += G) {
        const int t = base + sub;
        int c = 0;
        float v = 0.f;
        if (t < end) { c = col_idx[t]; v = alpha * val[t]; }
        const int cnt = min(G, end - base);
        for (int j = 0; j < cnt; j += 4) {
            int cj[4];
            float vj[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                cj[u] = __shfl(c, (j + u) & (G - 1), G);   // entries at or past cnt are never accumulated
                vj[u] = __shfl(v, (j + u) & (G - 1), G);
            }
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int unit = sub + it * G;
                if (unit * V::kVec < n) {
                    const int col0 = V::at(unit, n);
                    typename V::T x[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        x[u] = (j + u < cnt) ? V::load(B + (size_t)cj[u] * ldb + col0) : V::zero();
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (j + u < cnt) V::fma(acc[it], vj[u], RELU_IN ? V::relu(x[u]) : x[u]);
                }
            }
        }
    }

    if (row < m && !deferred && owner) {
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int unit = sub + it * G;
            if (unit * V::kVec < n) {
                const int col0 = V::at(unit, n);
                if (hub >= 0) acc[it] = V::axpby(V::zero(), alpha, hub_row_sum<V>(hubs.part + (size_t)hub * hubs.ld + col0, hubs.ld, entries, hubs.shift));
                V::update(C + (size_t)row * ldc, unit, n, acc[it], beta);
            }
        }
    }

    __syncthreads();
    const int nlong = lr_count;           // uniform across the workgroup
    const int width = G * V::kVec * ITERS;
    for (int li = 0; li < nlong; ++li) {
        const int lrow = lr_list[li];
        const int ls = row_ptr[lrow], le = row_ptr[lrow + 1];
#pragma unroll
        for (int it = 0; it < ITERS; ++it) acc[it] = V::zero();

        int t = ls + grp;
        for (; t + 3 * ngroups < le; t += 4 * ngroups) {
            int c4[4];
            float v4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { c4[u] = col_idx[t + u * ngroups]; v4[u] = alpha * val[t + u * ngroups]; }
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int unit = sub + it * G;
                if (unit * V::kVec < n) {
                    const int col0 = V::at(unit, n);
                    typename V::T x[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) x[u] = V::load(B + (size_t)c4[u] * ldb + col0);
#pragma unroll
                    for (int u = 0; u < 4; ++u) V::fma(acc[it], v4[u], RELU_IN ? V::relu(x[u]) : x[u]);
                }
            }
        }
        for (; t < le; t += ngroups) {
            const int c0 = col_idx[t];
            const float v0 = alpha * val[t];
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int unit = sub + it * G;
                if (unit * V::kVec < n) {
                    const int col0 = V::at(unit, n);
                    const typename V::T x = V::load(B + (size_t)c0 * ldb + col0);
                    V::fma(acc[it], v0, RELU_IN ? V::relu(x) : x);
                }
            }
        }

#pragma unroll
        for (int it = 0; it < ITERS; ++it)
            V::store(red + (size_t)grp * width + (sub + it * G) * V::kVec, acc[it]);
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int it = 0; it < ITERS; ++it) {
                const int unit = sub + it * G;
                if (unit * V::kVec < n) {
                    typename V::T s = V::zero();
                    for (int g = 0; g < ngroups; ++g) s = V::add(s, V::load(red + (size_t)g * width + unit * V::kVec));
                    V::update(C + (size_t)lrow * ldc, unit, n, s, beta);
                }
            }
        }
        __syncthreads();
    }
}

inline int ilog2_ceil(int x)
{
    int l = 0;
    while ((1 << l) < x) ++l;
    return l;
}

template <class V, int ITERS>
int launch_slab(int m, int n, float alpha, const int* row_ptr, const int* col_idx, const float* val,
                const float* B, int ldb, float beta, float* C, int ldc, int logG, const HubPlan& hubs, bool one_row, bool relu_in, hipStream_t s)
{
    const int groups_per_block = one_row ? 1 : kBlock >> logG;
    const unsigned blocks = ceil_div_u((size_t)m, (size_t)groups_per_block);
    auto kernel = relu_in ? spmm_rowgroup_kernel<V, ITERS, true, false> : spmm_rowgroup_kernel<V, ITERS, false, false>;
    if constexpr (ITERS == 1) {
        if ((1 << logG) <= kNarrowGroup) kernel = relu_in ? spmm_rowgroup_kernel<V, 1, true, true> : spmm_rowgroup_kernel<V, 1, false, true>;
    }
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kBlock), 0, s,
                       m, n, alpha, row_ptr, col_idx, val, B, ldb, beta, C, ldc, logG, one_row ? -1 : kLongRow, hubs);
    GNNHIP_LAUNCH_CHECK("spmm_rowgroup");
    return GNNHIP_OK;
}

}  // namespace

// Shared with the fused forward: C = alpha*A*B + beta*C on stream s.
int spmm_dispatch(int m, int k, int n, long long nnz, float alpha, const int* row_ptr, const int* col_idx, const float* val,
                  const float* B, int ldb, float beta, float* C, int ldc, hipStream_t s, bool reuse_plan,
                  CsrPlan* plan, bool relu_in)
{
    // large matrices with many entries per row (power-law graphs): rows cut into pieces, summed in column order.  That
    // route takes all its scratch (about 40 bytes per entry of A + 4 n bytes per piece) before its first launch: when
    // the device cannot give it, C is untouched and the row-group route below, which needs far less, does the product.
    if (int rc = spmm_pieces_dispatch(m, k, n, nnz, alpha, row_ptr, col_idx, val, B, ldb, beta, C, ldc, s, reuse_plan, plan, relu_in);
        rc != GNNHIP_EUNSUPPORTED && rc != GNNHIP_ENOMEM)
        return rc;
    return spmm_plain_dispatch(m, k, n, nnz, alpha, row_ptr, col_idx, val, B, ldb, beta, C, ldc, s, reuse_plan, plan ? &plan->row_hub : nullptr, relu_in);
}

// The row-group route alone (with its pass over very long rows); nnz may be an upper bound.  row_hub: where a plan's
// owner keeps the pass's arrays across calls.
int spmm_plain_dispatch(int m, int k, int n, long long nnz, float alpha, const int* row_ptr, const int* col_idx, const float* val,
                        const float* B, int ldb, float beta, float* C, int ldc, hipStream_t s, bool reuse_plan, HubStore* row_hub, bool relu_in)
{
    (void)k;
    // few rows of hundreds of entries each (sum-pooling into subgraphs): a workgroup per row instead of a lane group
    const bool one_row = m < kHubMinRows && nnz >= kOneRowMeanEntries * (long long)m;
    const bool vec4 = (n % 4 == 0) && (ldb % 4 == 0) && (ldc % 4 == 0) && aligned16(B) && aligned16(C);
    const int vec = n >= 4 ? 4 : 1;
    // columns are processed in slabs of at most 64 lanes * vec * 4
    const int slab_max = kWave * vec * 4;
    for (int col0 = 0; col0 < n; col0 += slab_max) {
        const int w = (n - col0 < slab_max) ? (n - col0) : slab_max;
        const bool one = w < 4;                             // also what n mod 1024 leaves behind the full slabs
        const int units = one ? w : (w + 3) / 4;            // column units of a lane
        int logG = ilog2_ceil(units < kWave ? units : kWave);
        const int G = 1 << logG;
        const int iters = (units + G - 1) / G;              // 1..4
        const float* Bs = B + col0;
        float* Cs = C + col0;
        int rc;
        HubPlan hubs;
        if ((rc = hub_prepass(m, w, nnz, row_ptr, col_idx, val, Bs, ldb, s, &hubs, reuse_plan && n <= slab_max, relu_in, kHubThreshold, kHubChunk, -1, row_hub))) return rc;
        if (one) {
            rc = launch_slab<ColsOne, 1>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
        } else if (vec4) {
            if (iters <= 1) rc = launch_slab<ColsWide, 1>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
            else if (iters == 2) rc = launch_slab<ColsWide, 2>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
            else rc = launch_slab<ColsWide, 4>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
        } else {
            if (iters <= 1) rc = launch_slab<ColsLoose, 1>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
            else if (iters == 2) rc = launch_slab<ColsLoose, 2>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
            else rc = launch_slab<ColsLoose, 4>(m, w, alpha, row_ptr, col_idx, val, Bs, ldb, beta, Cs, ldc, logG, hubs, one_row, relu_in, s);
        }
        if (rc) return rc;
    }
    return GNNHIP_OK;
}

}  // namespace gnnhip

using namespace gnnhip;

extern "C" int gnnhip_spmm_csr_f32(int m, int k, int n, int nnz, float alpha, const int* row_ptr, const int* col_idx,
                                   const float* val, const float* B, int ldb, float beta, float* C, int ldc,
                                   void* stream)
{
    GNNHIP_REQUIRE(m >= 0 && k >= 0 && n >= 0 && nnz >= 0, "negative dimension in spmm (m=%d k=%d n=%d nnz=%d)", m, k, n, nnz);
    if (m == 0 || n == 0) return GNNHIP_OK;
    GNNHIP_REQUIRE(row_ptr && C, "null row_ptr or output in spmm");
    GNNHIP_REQUIRE(ldb >= n && ldc >= n, "leading dimension smaller than n in spmm (ldb=%d ldc=%d n=%d)", ldb, ldc, n);
    GNNHIP_REQUIRE(k == 0 || B, "null dense operand in spmm");   // col_idx / val may be null when A has no entries
    if (int rc = require_ready()) return rc;
    return spmm_dispatch(m, k, n, nnz, alpha, row_ptr, col_idx, val, B, ldb, beta, C, ldc, as_stream(stream));
}

extern "C" int gnnhip_spmm_csr_planned_f32(void* plan, int n, float alpha, const float* B, int ldb, float beta, float* C, int ldc,
                                           void* stream)
{
    CsrPlan* p = as_csr_plan(plan);
    GNNHIP_REQUIRE(p, "%p is not a live CSR plan", plan);
    GNNHIP_REQUIRE(n >= 0, "negative width in spmm_csr_planned (n=%d)", n);
    if (p->m == 0 || n == 0) return GNNHIP_OK;
    GNNHIP_REQUIRE(C, "null output in spmm_csr_planned");
    GNNHIP_REQUIRE(ldb >= n && ldc >= n, "leading dimension smaller than n in spmm_csr_planned (ldb=%d ldc=%d n=%d)", ldb, ldc, n);
    GNNHIP_REQUIRE(p->k == 0 || B, "null dense operand in spmm_csr_planned");
    if (int rc = require_ready()) return rc;
    return spmm_dispatch(p->m, p->k, n, p->nnz, alpha, p->row_ptr, p->col_idx, p->val, B, ldb, beta, C, ldc, as_stream(stream), false, p);
}
