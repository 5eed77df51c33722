// Device-side grouping of (key, payload) pairs into CSR, and CSR transposition.
//
// graphnn builds the CSR operands of a batch on the host by walking per-node lists
// (src/nn/msg_pass.cpp:46-177); row i of such a matrix lists the payloads of the pairs
// whose key is i, in insertion order.  That is a stable sort of the pair indices by key.
// Here: a least-significant-digit radix sort (digits of 8, 10 or 11 bits, so that up to 4M rows
// take two passes) whose every pass is stable, then the row pointers from the sorted keys.
// A matrix and its transpose are grouped side by side in the same launches.
//
// One pass over n pairs, tiles of 2048 pairs per workgroup:
//   histogram   per tile, an LDS counter per digit -> hist[digit][tile]
//   scan        exclusive scan of hist in digit-major order
//   scatter     a wavefront takes 512 consecutive pairs of the tile, 64 at a time; lanes with
//               the same digit find each other with a ballot per bit, their rank is the running
//               count of that digit in the wavefront's segment plus the number of lower lanes;
//               segment counts are then prefixed over the four wavefronts.  Destination =
//               scanned hist[digit][tile] + rank.  Order inside a digit = input order: stable.
// No atomics on global memory; the result is a pure function of the input.
//
// At the sizes of training batches (10^5 to 10^6 pairs) a launch costs about what it does: 659,010 pairs on 299,536
// rows, both ways, took 36 launches and 206 us with 8-bit digits, one grouping after the other; 9 launches and
// 114 us now.
#include <algorithm>
#include <type_traits>

#include "gnnhip_internal.h"

namespace gnnhip {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kItems = 8;
constexpr int kTile = kBlock * kItems;          // 2048 pairs per workgroup
constexpr int kSeg = kTile / kWavesPerBlock;    // 512 consecutive pairs per wavefront

// What one grouping reads and writes, and its part of the scratch.
struct GroupJob {
    const int* key;                              // as the caller holds them, read by the first pass
    const int* payload;
    const float* val_in;                         // null: 1
    int key_stride, payload_stride;
    int* row_ptr;
    int* col_idx;
    float* val;
    unsigned *k0, *k1, *v0, *v1;                 // keys and pair indices, before and after a pass
    int *hist, *seg;
};
constexpr int kMaxJobs = 2;                      // blockIdx.y picks one
struct GroupJobs { GroupJob job[kMaxJobs]; };

// a key outside [0, rows) is a caller error, but it must not send the row-pointer kernels out of bounds
__device__ __forceinline__ unsigned first_key(const GroupJob& j, long long i, int rows) { return (unsigned)min(max(j.key[i * j.key_stride], 0), rows - 1); }

template <int BITS>
__device__ __forceinline__ void tile_histogram(int* h, int ntiles, int* __restrict__ hist)
{
    for (int d = threadIdx.x; d < (1 << BITS); d += kBlock) hist[(size_t)d * ntiles + blockIdx.x] = h[d];
}

// FIRST: the keys are the caller's
template <int BITS, bool FIRST>
__global__ __launch_bounds__(kBlock) void radix_hist_kernel(GroupJobs jobs, long long n, int rows, int shift, int ntiles)
{
    const GroupJob& j = jobs.job[blockIdx.y];
    __shared__ int h[1 << BITS];
    for (int d = threadIdx.x; d < (1 << BITS); d += kBlock) h[d] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * kTile;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const long long idx = base + i * kBlock + threadIdx.x;
        if (idx < n) atomicAdd(&h[((FIRST ? first_key(j, idx, rows) : j.k0[idx]) >> shift) & ((1 << BITS) - 1)], 1);
    }
    __syncthreads();
    tile_histogram<BITS>(h, ntiles, j.hist);
}

// ---- exclusive scan of an int array of any length: segment sums, scan of the sums, apply
//      A launch over a few hundred thousand elements is latency, so it takes many workgroups of one 128-bit word per lane (the
//      arrays start on one): segments of 1,024.  With segments of 4,096, sixteen strided loads per lane, 300,001 elements were
//      the work of 74 workgroups, 6.2 us to apply where it is 4.7 now.  What writes an array can add up its segments on the way
//      (scan_from_sums_i32), which saves the first launch, 4.8 us.
__device__ __forceinline__ int block_scan_256(int v, int* sh, int* total)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int incl = v;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(incl, d, kWave);
        if (lane >= d) incl += o;
    }
    if (lane == kWave - 1) sh[wave] = incl;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; ++w) {
        if (w < wave) base += sh[w];
        tot += sh[w];
    }
    __syncthreads();
    *total = tot;
    return base + incl - v;
}

struct ScanJobs { int* x[kMaxJobs]; int* seg[kMaxJobs]; };      // blockIdx.y picks one; all of the same length

// elements base .. base + 3 of x[n], 0 past the end
__device__ __forceinline__ int4 load_four(const int* __restrict__ x, long long base, long long n)
{
    if (base + 4 <= n) return *reinterpret_cast<const int4*>(x + base);
    return {base < n ? x[base] : 0, base + 1 < n ? x[base + 1] : 0, base + 2 < n ? x[base + 2] : 0, 0};
}

__global__ __launch_bounds__(kBlock) void scan_segment_sums_kernel(ScanJobs jobs, long long n)
{
    __shared__ int sh[kWavesPerBlock];
    const int4 v = load_four(jobs.x[blockIdx.y], (long long)blockIdx.x * kScanSeg + threadIdx.x * 4, n);
    int tot;
    block_scan_256(v.x + v.y + v.z + v.w, sh, &tot);
    if (threadIdx.x == 0) jobs.seg[blockIdx.y][blockIdx.x] = tot;
}

// one workgroup: exclusive scan of the nseg segment sums in place
__global__ __launch_bounds__(1024) void scan_small_kernel(ScanJobs jobs, int nseg)
{
    int* __restrict__ x = jobs.seg[blockIdx.y];
    __shared__ int wave_tot[1024 / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int per = (nseg + 1023) / 1024;
    const int lo = min(tid * per, nseg), hi = min(lo + per, nseg);
    int local = 0;
    for (int i = lo; i < hi; ++i) local += x[i];
    int incl = local;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(incl, d, kWave);
        if (lane >= d) incl += o;
    }
    if (lane == kWave - 1) wave_tot[wave] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; ++w) base += wave_tot[w];
    int run = base + incl - local;
    for (int i = lo; i < hi; ++i) { const int v = x[i]; x[i] = run; run += v; }
}

// SUMS: seg holds the segments' sums and the workgroup adds up those before its own; else their scan
template <bool SUMS>
__global__ __launch_bounds__(kBlock) void scan_apply_kernel(ScanJobs jobs, long long n)
{
    int* __restrict__ x = jobs.x[blockIdx.y];
    const int* __restrict__ seg = jobs.seg[blockIdx.y];
    __shared__ int sh[kWavesPerBlock];
    const long long base = (long long)blockIdx.x * kScanSeg + threadIdx.x * 4;
    int ahead = 0;
    if (SUMS) {
        for (int i = threadIdx.x; i < (int)blockIdx.x; i += kBlock) ahead += seg[i];
    }
    const int4 v = load_four(x, base, n);
    int tot;
    if (SUMS) block_scan_256(ahead, sh, &ahead);
    else ahead = seg[blockIdx.x];
    const int run = ahead + block_scan_256(v.x + v.y + v.z + v.w, sh, &tot);
    const int4 o = {run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z};
    if (base + 4 <= n) {
        *reinterpret_cast<int4*>(x + base) = o;
    } else {
        if (base < n) x[base] = o.x;
        if (base + 1 < n) x[base + 1] = o.y;
        if (base + 2 < n) x[base + 2] = o.z;
    }
}

// Up to here (2M elements) a workgroup adds up the segments itself; beyond, a launch of one workgroup scans the sums first.  With segments of 4,096
// the line was at 8M, and between the two the smaller segments are still ahead: grouping 20,000,000 pairs, counters of 2.5M, 1,829 -> 1,780 us, a
// transpose of 24,000,000 entries 3,720 -> 3,667.
constexpr int kSumsMaxSegments = 2048;

// SUMMED: the segments' sums are there already
template <bool SUMMED = false>
int exclusive_scans(int count, const ScanJobs& jobs, long long n, hipStream_t s)
{
    if (n <= 0) return GNNHIP_OK;
    const int nseg = (int)scan_seg_ints(n);
    if (!SUMMED) hipLaunchKernelGGL(scan_segment_sums_kernel, dim3(nseg, count), dim3(kBlock), 0, s, jobs, n);
    if (nseg <= kSumsMaxSegments) {
        hipLaunchKernelGGL(scan_apply_kernel<true>, dim3(nseg, count), dim3(kBlock), 0, s, jobs, n);
    } else {
        hipLaunchKernelGGL(scan_small_kernel, dim3(1, count), dim3(1024), 0, s, jobs, nseg);
        hipLaunchKernelGGL(scan_apply_kernel<false>, dim3(nseg, count), dim3(kBlock), 0, s, jobs, n);
    }
    GNNHIP_LAUNCH_CHECK("exclusive_scan_i32");
    return GNNHIP_OK;
}

}  // namespace

// Exclusive scan of x[n], which starts on a 128-bit word, from the sums of its segments of kScanSeg elements in seg[scan_seg_ints(n)]
// (what writes an array adds up its segments at no cost: a launch of 4.8 us saved per array).  seg is overwritten.
int scan_from_sums_i32(int* x, long long n, int* seg, hipStream_t s)
{
    return exclusive_scans<true>(1, ScanJobs{{x, nullptr}, {seg, nullptr}}, n, s);
}

// two arrays of n elements in the same launches; the second one's sums follow the first one's
int scan_pair_from_sums_i32(int* x, int* y, long long n, int* seg, hipStream_t s)
{
    return exclusive_scans<true>(2, ScanJobs{{x, y}, {seg, seg + scan_seg_ints(n)}}, n, s);
}

namespace {

// FIRST: the keys are the caller's and a pair's value is its index
template <int BITS, bool FIRST>
__global__ __launch_bounds__(kBlock) void radix_scatter_kernel(GroupJobs jobs, long long n, int rows, int shift, int ntiles)
{
    constexpr int kDigits = 1 << BITS;
    const GroupJob& j = jobs.job[blockIdx.y];
    const int* __restrict__ hist_scanned = j.hist;
    __shared__ int cnt[kWavesPerBlock][kDigits];      // running, then total, count of each digit per wavefront segment
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    for (int i = threadIdx.x; i < kWavesPerBlock * kDigits; i += kBlock) (&cnt[0][0])[i] = 0;
    __syncthreads();

    const long long seg0 = (long long)blockIdx.x * kTile + wave * kSeg;
    unsigned k[kItems], v[kItems];
    int rank[kItems];
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const long long idx = seg0 + i * kWave + lane;
        const bool live = idx < n;
        k[i] = !live ? 0u : FIRST ? first_key(j, idx, rows) : j.k0[idx];
        v[i] = !live ? 0u : FIRST ? (unsigned)idx : j.v0[idx];
        const unsigned d = (k[i] >> shift) & (kDigits - 1);
        // lanes of this round with the same digit (dead lanes match nobody)
        unsigned long long same = __ballot(live);
#pragma unroll
        for (int b = 0; b < BITS; ++b) {
            const unsigned long long bal = __ballot((d >> b) & 1u);
            same &= ((d >> b) & 1u) ? bal : ~bal;
        }
        int r = 0;
        if (live) {
            const int before = cnt[wave][d];                       // every lane of the group reads before its leader writes
            r = before + __popcll(same & below);
            if ((same & below) == 0) cnt[wave][d] = before + __popcll(same);
        }
        rank[i] = r;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    __syncthreads();
    // prefix of the segment counts over the wavefronts, per digit
    for (int d = threadIdx.x; d < kDigits; d += kBlock) {
        int run = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) { const int c = cnt[w][d]; cnt[w][d] = run; run += c; }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const long long idx = seg0 + i * kWave + lane;
        if (idx < n) {
            const unsigned d = (k[i] >> shift) & (kDigits - 1);
            const long long dst = (long long)hist_scanned[(size_t)d * ntiles + blockIdx.x] + cnt[wave][d] + rank[i];
            j.k1[dst] = k[i];
            j.v1[dst] = v[i];
        }
    }
}

// row_ptr from the sorted keys: position i opens every row in (key[i-1], key[i]]; the last position closes the rest
__device__ __forceinline__ void open_rows(const GroupJob& j, long long i, long long n, int rows)
{
    const long long k = j.k0[i];
    const long long kprev = (i == 0) ? -1 : (long long)j.k0[i - 1];
    for (long long r = kprev + 1; r <= k; ++r) j.row_ptr[r] = (int)i;
    if (i == n - 1)
        for (long long r = k + 1; r <= rows; ++r) j.row_ptr[r] = (int)n;
}

__global__ __launch_bounds__(kBlock) void empty_rows_kernel(GroupJobs jobs, int rows)
{
    const long long r = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (r <= rows) jobs.job[blockIdx.y].row_ptr[r] = 0;
}

__global__ __launch_bounds__(kBlock) void row_ptr_from_sorted_kernel(GroupJobs jobs, long long n, int rows)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) open_rows(jobs.job[blockIdx.y], i, n, rows);
}

// AVERAGE: values 1 / row length, which wait for the finished row pointers; otherwise the row pointers are formed here too
template <bool AVERAGE>
__global__ __launch_bounds__(kBlock) void fill_grouped_kernel(GroupJobs jobs, long long n, int rows)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const GroupJob& j = jobs.job[blockIdx.y];
    const unsigned src = j.v0[i];
    j.col_idx[i] = j.payload[(long long)src * j.payload_stride];
    float w = j.val_in ? j.val_in[src] : 1.0f;
    if (AVERAGE) {
        const unsigned r = j.k0[i];
        w = (float)(1.0 / (double)(j.row_ptr[r + 1] - j.row_ptr[r]));      // as the reference: double divide, then narrowed
    }
    j.val[i] = w;
    if (!AVERAGE) open_rows(j, i, n, rows);
}

// row index of every entry of a CSR matrix
__global__ __launch_bounds__(kBlock) void expand_rows_kernel(int m, const int* __restrict__ row_ptr, int* __restrict__ row_of)
{
    const int lane = threadIdx.x & (kWave - 1);
    const long long row = ((long long)blockIdx.x * kBlock + threadIdx.x) / kWave;
    if (row >= m) return;
    const int a = row_ptr[row], b = row_ptr[row + 1];
    for (int t = a + lane; t < b; t += kWave) row_of[t] = (int)row;
}

// ---- small inputs: the whole grouping in one launch ----
// A batch of a few hundred small graphs is latency, not bandwidth: the dozen launches of the radix passes
// cost more than the host loop they replace.  One launch of up to 64 workgroups instead.  The rows are cut
// into as many runs; every workgroup reads ALL keys (they are a few L2 lines per lane) and keeps the pairs
// of its own run of rows, so no workgroup ever waits for another: the number of keys below its first row,
// which it counts on the way, is where its part of the result starts.  Between the first read of the keys
// and the last write of the result everything is in LDS:
//   lengths    LDS counters (atomics), the pairs below the run, and a check whether the keys already ascend
//   scan       row_ptr; the counters become cursors
//   place      every pair takes the next slot of its row in whatever order the hardware serves the
//              atomics; the slot (16 bits, in LDS) keeps the pair's INDEX, so that the next step can put
//              every row into input order again.  Ascending keys: the pairs of the run are consecutive
//              and in order already, nothing to place or to order.
//   order      rows of up to 8 entries: a thread sorts them in registers (a fixed network);
//              up to 64: a lane of a wavefront holds an entry and counts the smaller ones;
//              longer rows: a wavefront marks the row's pair indices in a bitmap of its own and reads
//              the set bits back in ascending order, 64 words at a time (a prefix sum of the
//              population counts gives every word its first slot)
//   write      slot after slot, coalesced: payload (and value) of the pair the slot names
// Keys are read four to a load (where they are not strided), all of a thread's sixteen before the first is used.  What bounds it is
// the chain of these steps: 16,380 pairs of 7,450 rows take 3 us to read and count, 0.9 to scan, 0.7 to place, 0.7 to order and
// 1.5 to write, behind the 4 of any launch with much LDS (both ways at once 16.5 -> 9.5 us; 16 workgroups of 1,024 lanes with a
// key per load before).  More, smaller workgroups shorten every step but the reading (6,175 pairs 11.4 -> 7.6, 60,000 49 -> 24 us);
// rows of 9 to 64 entries cost 80 to 700 us per 65,000 pairs when each walked a bitmap.  By rank such a row takes a third of a
// microsecond of a SIMD's instructions, so few rows are spread over many workgroups: runs of 8 rows, and 8 wavefronts at least (2,000 pairs of 66 rows:
// runs of 64 rows and 4 wavefronts 27 us, of 16 rows 13, of 8 rows and 8 wavefronts 7.9).  The order of the entries is a
// pure function of the input, as on the radix route.  Sizes: 4 bytes per row of a run, 2 per pair, one
// bitmap of n bits (as many as fit, up to one per wavefront) in 160 KB of LDS; at most 65,536 pairs.
constexpr int kSmallPairs = 1 << 16;
constexpr int kSmallShort = 8;
constexpr int kSmallBatch = 16;
constexpr int kSmallLdsInts = 160 * 1024 / 4;
constexpr int kSmallMisc = 48;
constexpr int kSmallGroups = 64;           // workgroups at most, per grouping
constexpr int kSmallRunRows = 8;           // rows per workgroup at least

struct SmallLayout {
    int block;                            // lanes per workgroup
    int groups, run;                      // workgroups, rows per workgroup (a multiple of kSmallRunRows)
    int slots, longs, misc, bitmaps;      // offsets in ints (the counters start at 0)
    int words, nbitmaps;                  // words per bitmap, number of bitmaps
};
// false: the input does not fit the workgroups' LDS
inline bool small_layout(long long rows, long long n, SmallLayout* out)
{
    if (n < 1 || n > kSmallPairs || rows < 1) return false;
    SmallLayout l;
    long long groups = (rows + kSmallRunRows - 1) / kSmallRunRows;
    if (groups > kSmallGroups) groups = kSmallGroups;
    const long long run = ((rows + groups - 1) / groups + kSmallRunRows - 1) / kSmallRunRows * kSmallRunRows;
    if (run > kSmallLdsInts) return false;
    l.run = (int)run;
    l.groups = (int)((rows + run - 1) / run);
    l.slots = l.run;
    l.longs = l.slots + (int)((n + 1) / 2);
    l.misc = l.longs + (int)((n / (kSmallShort + 1) + 2) / 2);
    l.bitmaps = l.misc + kSmallMisc;
    l.words = (int)((n + 31) / 32);
    const int room = kSmallLdsInts - l.bitmaps;
    if (room < l.words) return false;
    // the keys in one batch of loads where that can be, four rows of the run per lane at most
    const long long per_lane = std::max((n + kSmallBatch - 1) / kSmallBatch, run / 4);
    l.block = per_lane <= 512 ? 512 : 1024;
    const int waves = l.block / kWave;
    l.nbitmaps = room / l.words < waves ? room / l.words : waves;
    *out = l;
    return true;
}

__device__ __forceinline__ void order_pair(int& a, int& b)
{
    const int lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}

// One grouping of the n pairs.  A launch carries one or two of them (the same pairs grouped by either member:
// a matrix and its transpose); workgroup b works on job b / groups.
struct SmallJob {
    const int* key;
    const int* payload;
    const float* val_in;
    int* row_ptr;
    int* col_idx;
    float* val;
    int key_stride, payload_stride;
};

// DENSE: keys follow each other in memory
template <int BLOCK, bool DENSE>
__global__ __launch_bounds__(BLOCK) void csr_group_small_kernel(int rows, int n, SmallLayout lay, SmallJob job0, SmallJob job1, int average)
{
    constexpr int kWaves = BLOCK / kWave;
    const bool second = (int)blockIdx.x >= lay.groups;
    const int run_index = (int)blockIdx.x - (second ? lay.groups : 0);
    const int* __restrict__ key = second ? job1.key : job0.key;
    const int* __restrict__ payload = second ? job1.payload : job0.payload;
    const float* __restrict__ val_in = second ? job1.val_in : job0.val_in;
    int* __restrict__ row_ptr = second ? job1.row_ptr : job0.row_ptr;
    int* __restrict__ col_idx = second ? job1.col_idx : job0.col_idx;
    float* __restrict__ val = second ? job1.val : job0.val;
    const int key_stride = second ? job1.key_stride : job0.key_stride;
    const int payload_stride = second ? job1.payload_stride : job0.payload_stride;
    extern __shared__ int small_lds[];
    int* cnt = small_lds;                          // one per row of this workgroup's run
    unsigned short* slots = reinterpret_cast<unsigned short*>(small_lds + lay.slots);
    unsigned short* longs = reinterpret_cast<unsigned short*>(small_lds + lay.longs);       // rows of more than kSmallShort entries
    int* misc = small_lds + lay.misc;              // [0] long rows, [1] keys out of order, [2..17] wavefront totals, [18..33] pairs below
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    const int top = rows - 1;
    const int lo = run_index * lay.run, mine = min(lay.run, rows - lo);            // this run: rows lo .. lo + mine - 1

    for (int r = tid; r < mine; r += BLOCK) cnt[r] = 0;
    if (tid < kSmallMisc) misc[tid] = 0;
    __syncthreads();

    // lengths.  DENSE: a lane takes four consecutive pairs at a time and counts equal neighbours among them together.  Else the loads
    // of four pairs a lane would each spread over four times as many lines (60,000 pairs of two ints: 58 us, 39 so): lanes hold consecutive
    // pairs, and a run of equal keys is counted by its first lane alone.  The keys of the first batch stay in registers for `place`.
    bool disorder = false;
    int below = 0;
    int first_keys[kSmallBatch];
    const bool words = DENSE && (reinterpret_cast<size_t>(key) & 15) == 0;
    auto pair_of = [&](int base, int u) { return base + (DENSE ? ((u / 4) * BLOCK + tid) * 4 + (u & 3) : u * BLOCK + tid); };
    auto load_keys = [&](int base, int (&k)[kSmallBatch]) {       // clamped; -1 past the last pair
        if constexpr (DENSE) {
#pragma unroll
            for (int v = 0; v < kSmallBatch / 4; ++v) {
                const int e = pair_of(base, 4 * v);
                int4 x = make_int4(-1, -1, -1, -1);
                if (words && e + 3 < n) {
                    x = *reinterpret_cast<const int4*>(key + e);
                } else {
                    if (e + 0 < n) x.x = key[e + 0];
                    if (e + 1 < n) x.y = key[e + 1];
                    if (e + 2 < n) x.z = key[e + 2];
                    if (e + 3 < n) x.w = key[e + 3];
                }
                k[4 * v] = x.x; k[4 * v + 1] = x.y; k[4 * v + 2] = x.z; k[4 * v + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int u = 0; u < kSmallBatch; ++u) {
                const int e = pair_of(base, u);
                k[u] = e < n ? key[(long long)e * key_stride] : -1;
            }
        }
#pragma unroll
        for (int u = 0; u < kSmallBatch; ++u) k[u] = pair_of(base, u) < n ? min(max(k[u], 0), top) : -1;
    };
    for (int base = 0; base < n; base += BLOCK * kSmallBatch) {       // every lane walks every batch: the shuffles need them
        constexpr int kEach = DENSE ? 4 : 1;                      // consecutive pairs of a lane
        int k[kSmallBatch], before[kSmallBatch / kEach];
#pragma unroll
        for (int v = 0; v < kSmallBatch / kEach; ++v) {
            const int e = pair_of(base, kEach * v);
            before[v] = lane == 0 && e > 0 && e < n ? key[(long long)(e - 1) * key_stride] : -1;
        }
        load_keys(base, k);
#pragma unroll
        for (int v = 0; v < kSmallBatch / kEach; ++v) {
            const int left = __shfl_up(k[kEach * v + kEach - 1], 1, kWave);
            int prev = lane == 0 ? (before[v] < 0 ? before[v] : min(before[v], top)) : left;
            if constexpr (DENSE) {
                int run = 1;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int kk = k[4 * v + j];
                    if (base == 0) first_keys[4 * v + j] = kk;
                    disorder |= kk >= 0 && prev > kk;
                    below += kk >= 0 && kk < lo;
                    prev = kk;
                    if (j < 3 && k[4 * v + (j < 3 ? j + 1 : 3)] == kk) {
                        ++run;
                    } else {
                        if (kk >= 0 && (unsigned)(kk - lo) < (unsigned)mine) atomicAdd(&cnt[kk - lo], run);
                        run = 1;
                    }
                }
            } else {
                const int kk = k[v];
                if (base == 0) first_keys[v] = kk;
                disorder |= kk >= 0 && prev > kk;
                below += kk >= 0 && kk < lo;
                const bool head = lane == 0 || left != kk;
                const unsigned long long heads = __ballot(head);
                if (head && kk >= 0 && (unsigned)(kk - lo) < (unsigned)mine) {
                    const unsigned long long later = lane == kWave - 1 ? 0ull : heads >> (lane + 1);
                    atomicAdd(&cnt[kk - lo], later ? __ffsll((long long)later) : kWave - lane);
                }
            }
        }
    }
    if (disorder) misc[1] = 1;
    below = wave_sum_i(below);
    if (lane == 0) misc[18 + uwave] = below;
    __syncthreads();

    // exclusive scan: a wavefront owns a stretch of the run and walks it 64 rows at a time
    const int seg = ((mine + kWaves - 1) / kWaves + kWave - 1) & ~(kWave - 1);
    const int s0 = min(uwave * seg, mine), s1 = min(s0 + seg, mine);
    int part = 0;
    for (int r = s0 + lane; r < s1; r += kWave) part += cnt[r];
    part = wave_sum_i(part);
    if (lane == 0) misc[2 + uwave] = part;
    __syncthreads();
    const int upto = wave_inclusive_scan_i(lane < kWaves ? misc[2 + lane] : 0);
    const int first_slot = wave_sum_i(lane < kWaves ? misc[18 + lane] : 0);      // pairs of the runs before this one
    const int held = __builtin_amdgcn_readlane(upto, kWaves - 1);                 // pairs of this run
    int carry = uwave ? __builtin_amdgcn_readlane(upto, uwave - 1) : 0;
    for (int r = s0 + lane; r - lane < s1; r += kWave) {
        const int c = r < s1 ? cnt[r] : 0;
        const int through = wave_inclusive_scan_i(c);
        if (r < s1) cnt[r] = carry + through - c;
        carry += __builtin_amdgcn_readlane(through, kWave - 1);
    }
    const bool ascending = misc[1] == 0;
    __syncthreads();
    for (int r = tid; r < mine; r += BLOCK) row_ptr[lo + r] = first_slot + cnt[r];
    if (lo + mine == rows && tid == 0) row_ptr[rows] = n;

    if (!ascending) {
        __syncthreads();                  // the starts are on their way out; the counters turn into cursors
        auto place = [&](int base, const int (&k)[kSmallBatch]) {
#pragma unroll
            for (int u = 0; u < kSmallBatch; ++u) {
                const int r = k[u] - lo;                  // -1: past the last pair, outside every run
                if (k[u] >= 0 && (unsigned)r < (unsigned)mine) slots[atomicAdd(&cnt[r], 1)] = (unsigned short)pair_of(base, u);
            }
        };
        place(0, first_keys);
        for (int base = BLOCK * kSmallBatch; base < n; base += BLOCK * kSmallBatch) {
            int k[kSmallBatch];
            load_keys(base, k);
            place(base, k);
        }
        __syncthreads();                  // cnt[r] is now the end of row r

        for (int r0 = 0; r0 < mine; r0 += BLOCK) {
            const int r = r0 + tid;
            int a = 0, len = 0;
            if (r < mine) {
                a = r ? cnt[r - 1] : 0;
                len = cnt[r] - a;
            }
            if (len > kSmallShort) {
                longs[atomicAdd(&misc[0], 1)] = (unsigned short)r;
                len = 0;
            }
            if (__ballot(len >= 2) == 0ull) continue;
            if (__ballot(len > 4) == 0ull) {
                // nobody in this wavefront has more than 4: 5 exchanges order 4 values
                int v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = j < len ? (int)slots[a + j] : 0x7fffffff;
                order_pair(v[0], v[1]); order_pair(v[2], v[3]); order_pair(v[0], v[2]); order_pair(v[1], v[3]); order_pair(v[1], v[2]);
                if (len >= 2) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (j < len) slots[a + j] = (unsigned short)v[j];
                }
                continue;
            }
            int v[kSmallShort];
#pragma unroll
            for (int j = 0; j < kSmallShort; ++j) v[j] = j < len ? (int)slots[a + j] : 0x7fffffff;
            // 19 exchanges order 8 values
            order_pair(v[0], v[1]); order_pair(v[2], v[3]); order_pair(v[4], v[5]); order_pair(v[6], v[7]);
            order_pair(v[0], v[2]); order_pair(v[1], v[3]); order_pair(v[4], v[6]); order_pair(v[5], v[7]);
            order_pair(v[1], v[2]); order_pair(v[5], v[6]); order_pair(v[0], v[4]); order_pair(v[3], v[7]);
            order_pair(v[1], v[5]); order_pair(v[2], v[6]);
            order_pair(v[1], v[4]); order_pair(v[3], v[6]);
            order_pair(v[2], v[4]); order_pair(v[3], v[5]);
            order_pair(v[3], v[4]);
            if (len >= 2) {
#pragma unroll
                for (int j = 0; j < kSmallShort; ++j)
                    if (j < len) slots[a + j] = (unsigned short)v[j];
            }
        }
        __syncthreads();

        const int nlong = misc[0];
        // up to 64 entries: a lane holds one and counts the smaller ones (the values are distinct)
        for (int q = uwave; q < nlong; q += kWaves) {
            const int r = longs[q];
            const int a = r ? cnt[r - 1] : 0, len = cnt[r] - a;
            if (len > kWave) continue;
            const int v = lane < len ? (int)slots[a + lane] : kSmallPairs;
            const int ulen = __builtin_amdgcn_readfirstlane(len);
            int rank = 0;
            for (int j0 = 0; j0 < ulen; j0 += 8) {        // (a lane past the row holds what is larger than any entry)
#pragma unroll
                for (int j = 0; j < 8; ++j) rank += __builtin_amdgcn_readlane(v, j0 + j) < v;
            }
            if (lane < len) slots[a + rank] = (unsigned short)v;
        }
        if (nlong > 0 && wave < lay.nbitmaps) {
            unsigned* bits = reinterpret_cast<unsigned*>(small_lds + lay.bitmaps) + wave * lay.words;
            for (int i = lane; i < lay.words; i += kWave) bits[i] = 0u;
            for (int q = wave; q < nlong; q += lay.nbitmaps) {
                const int r = longs[q];
                const int a = r ? cnt[r - 1] : 0, b = cnt[r];
                if (b - a <= kWave) continue;
                int first = 0x7fffffff, last = -1;
                for (int i = a + lane; i < b; i += kWave) {
                    const int e = slots[i];
                    atomicOr(&bits[e >> 5], 1u << (e & 31));
                    first = min(first, e);
                    last = max(last, e);
                }
#pragma unroll
                for (int d = 1; d < kWave; d <<= 1) {
                    first = min(first, __shfl_xor(first, d, kWave));
                    last = max(last, __shfl_xor(last, d, kWave));
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const int last_word = last >> 5;
                int slot = a;
                for (int word0 = first >> 5; word0 <= last_word; word0 += kWave) {
                    const int word = word0 + lane;
                    unsigned m = 0u;
                    if (word <= last_word) {
                        m = bits[word];
                        bits[word] = 0u;
                    }
                    const int c = __popc(m);
                    const int through = wave_inclusive_scan_i(c);
                    int at = slot + through - c;
                    while (m) {
                        slots[at++] = (unsigned short)(word * 32 + (__ffs((int)m) - 1));
                        m &= m - 1u;
                    }
                    slot += __shfl(through, kWave - 1, kWave);
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        __syncthreads();
    }

    // slot i of this run holds pair e and is entry first_slot + i of the result: out it goes
    for (int base = tid; base < held; base += BLOCK * kSmallBatch) {
        int e[kSmallBatch], pay[kSmallBatch], k[kSmallBatch];
        float w[kSmallBatch];
#pragma unroll
        for (int u = 0; u < kSmallBatch; ++u) {
            const int i = base + u * BLOCK;
            e[u] = i < held ? (ascending ? first_slot + i : (int)slots[i]) : 0;
        }
#pragma unroll
        for (int u = 0; u < kSmallBatch; ++u) {
            const bool live = base + u * BLOCK < held;
            pay[u] = live ? payload[(long long)e[u] * payload_stride] : 0;
            w[u] = (live && val_in) ? val_in[e[u]] : 1.0f;
            k[u] = (live && average) ? key[(long long)e[u] * key_stride] : 0;
        }
#pragma unroll
        for (int u = 0; u < kSmallBatch; ++u) {
            const int i = base + u * BLOCK;
            if (i >= held) continue;
            if (average) {
                const int r = min(max(k[u], 0), top) - lo;
                const int len = ascending ? (r + 1 < mine ? cnt[r + 1] : held) - cnt[r] : cnt[r] - (r ? cnt[r - 1] : 0);
                w[u] = (float)(1.0 / (double)len);       // as the reference: double divide, then narrowed
            }
            col_idx[first_slot + i] = pay[u];
            val[first_slot + i] = w[u];
        }
    }
}

// col_idx[j] = j and val[j] = 1 (or 1 / row length) for j in [row_ptr[i], row_ptr[i+1]): a wavefront per row
// (row_ptr may be pinned host memory: then row_ptr_out, device memory, receives a copy for the kernels that follow)
__global__ __launch_bounds__(kBlock) void consecutive_rows_kernel(int rows, const int* __restrict__ row_ptr, int average,
                                                                  int* __restrict__ col_idx, float* __restrict__ val,
                                                                  int* __restrict__ row_ptr_out)
{
    const int lane = threadIdx.x & (kWave - 1);
    const long long row = ((long long)blockIdx.x * kBlock + threadIdx.x) / kWave;
    if (row >= rows) return;
    const int a = row_ptr[row], b = row_ptr[row + 1];
    if (row_ptr_out && lane == 0) {
        row_ptr_out[row] = a;
        if (row == rows - 1) row_ptr_out[rows] = b;
    }
    const float w = (average && b > a) ? (float)(1.0 / (double)(b - a)) : 1.0f;       // as the reference: double divide, then narrowed
    for (int j = a + lane; j < b; j += kWave) {
        col_idx[j] = j;
        val[j] = w;
    }
}

inline size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

}  // namespace

// order[i] = index of the key that comes i-th when n keys of `bits` bits (8 and 11: one pass of the radix sort, 16: two) are put in
// order, equal keys in input order.  keys, keys_out and spare are overwritten.  hist needs radix_hist_ints(n) ints, seg
// radix_seg_ints(n).
size_t radix_hist_ints(long long n) { return ((size_t)1 << 11) * (size_t)((n + kTile - 1) / kTile > 0 ? (n + kTile - 1) / kTile : 1); }
size_t radix_seg_ints(long long n) { return scan_seg_ints((long long)radix_hist_ints(n)); }

namespace {

template <int BITS>
int radix_pass(int count, const GroupJobs& jobs, bool first, long long n, int rows, int shift, hipStream_t s)
{
    const int ntiles = (int)((n + kTile - 1) / kTile);
    const dim3 grid(ntiles, count);
    if (first) hipLaunchKernelGGL((radix_hist_kernel<BITS, true>), grid, dim3(kBlock), 0, s, jobs, n, rows, shift, ntiles);
    else hipLaunchKernelGGL((radix_hist_kernel<BITS, false>), grid, dim3(kBlock), 0, s, jobs, n, rows, shift, ntiles);
    ScanJobs scans{};
    for (int i = 0; i < count; ++i) { scans.x[i] = jobs.job[i].hist; scans.seg[i] = jobs.job[i].seg; }
    if (int rc = exclusive_scans(count, scans, (long long)(1 << BITS) * ntiles, s)) return rc;
    if (first) hipLaunchKernelGGL((radix_scatter_kernel<BITS, true>), grid, dim3(kBlock), 0, s, jobs, n, rows, shift, ntiles);
    else hipLaunchKernelGGL((radix_scatter_kernel<BITS, false>), grid, dim3(kBlock), 0, s, jobs, n, rows, shift, ntiles);
    GNNHIP_LAUNCH_CHECK("radix pass");
    return GNNHIP_OK;
}

}  // namespace

int radix_order(unsigned* keys, int bits, long long n, unsigned* keys_out, unsigned* spare, unsigned* order, int* hist, int* seg, hipStream_t s)
{
    if (n <= 0) return GNNHIP_OK;
    GroupJobs jobs{};
    GroupJob& j = jobs.job[0];
    j.key = reinterpret_cast<const int*>(keys);                  // `bits` bits: never clamped
    j.key_stride = 1;
    j.k1 = keys_out;
    j.hist = hist; j.seg = seg;
    if (bits <= 11) {
        j.v1 = order;
        return bits <= 8 ? radix_pass<8>(1, jobs, true, n, 1 << 8, 0, s) : radix_pass<11>(1, jobs, true, n, 1 << 11, 0, s);
    }
    j.v1 = spare;
    if (int rc = radix_pass<8>(1, jobs, true, n, 1 << 16, 0, s)) return rc;
    j.k0 = keys_out; j.v0 = spare;
    j.k1 = keys; j.v1 = order;
    return radix_pass<8>(1, jobs, false, n, 1 << 16, 8, s);
}

// The one-launch grouping where it fits; false: it does not (nothing launched).  With t_row_ptr the same launch
// also groups the pairs by payload with the key as the payload: the transpose, its entries in pair order, values 1.
bool csr_group_small(int rows, long long n, const int* key, int key_stride, const int* payload, int payload_stride, const float* val_in,
                     int average, int* row_ptr, int* col_idx, float* val, int* t_row_ptr, int* t_col_idx, float* t_val, hipStream_t s)
{
    SmallLayout lay;
    if (!small_layout(rows, n, &lay)) return false;
    const SmallJob job0 = {key, payload, val_in, row_ptr, col_idx, val, key_stride, payload_stride};
    const SmallJob job1 = {payload, key, nullptr, t_row_ptr, t_col_idx, t_val, payload_stride, key_stride};
    const dim3 grid(lay.groups * (t_row_ptr ? 2 : 1));
    const size_t lds = sizeof(int) * (size_t)(lay.bitmaps + lay.words * lay.nbitmaps);
    auto launch = [&](auto block, auto dense) {
        constexpr int kSize = decltype(block)::value;
        constexpr bool kDense = decltype(dense)::value;
        static LdsLimit limit;
        if (limit.raise(reinterpret_cast<const void*>(csr_group_small_kernel<kSize, kDense>), sizeof(int) * kSmallLdsInts) != hipSuccess) return false;
        hipLaunchKernelGGL((csr_group_small_kernel<kSize, kDense>), grid, dim3(kSize), lds, s, rows, (int)n, lay, job0, job1, average);
        return true;
    };
    auto by_stride = [&](auto block) {
        const bool dense = key_stride == 1 && (!t_row_ptr || payload_stride == 1);
        return dense ? launch(block, std::true_type()) : launch(block, std::false_type());
    };
    if (lay.block == 512) return by_stride(std::integral_constant<int, 512>());
    return by_stride(std::integral_constant<int, 1024>());
}

inline int last_launch_status(const char* what)
{
    GNNHIP_LAUNCH_CHECK(what);
    return GNNHIP_OK;
}

// Groups n pairs by key (0 <= key < rows) keeping input order inside a group, `count` groupings side by side:
//   row_ptr[rows + 1], col_idx[i] = payload of the i-th pair in grouped order,
//   val[i] = val_in of that pair (or 1), or 1 / group size when average is set.
// key / payload are read with the given strides (in ints).  Uses scratch slot 0 of the stream.
int csr_group_pairs(int count, GroupJobs jobs, int rows, long long n, int average, hipStream_t s)
{
    if (n == 0) {
        hipLaunchKernelGGL(empty_rows_kernel, dim3((unsigned)(((long long)rows + kBlock) / kBlock), count), dim3(kBlock), 0, s, jobs, rows);
        GNNHIP_LAUNCH_CHECK("csr_group_pairs");
        return GNNHIP_OK;
    }
    int bits = 1;
    while (bits < 31 && (1ll << bits) < (long long)rows) ++bits;
    // two passes up to 4M rows: the narrowest digits that do it (the counters of a digit per tile are one more array to scan)
    const int digit = bits <= 16 ? 8 : bits <= 20 ? 10 : bits <= 22 ? 11 : 8;
    const int ntiles = (int)((n + kTile - 1) / kTile);
    const size_t nhist = ((size_t)1 << digit) * ntiles;
    size_t off = 0;
    auto carve = [&](size_t bytes) { const size_t o = off; off = round_up(off + bytes, 256); return o; };
    size_t o[kMaxJobs][6];
    for (int i = 0; i < count; ++i) {
        for (int a = 0; a < 4; ++a) o[i][a] = carve(sizeof(unsigned) * (size_t)n);
        o[i][4] = carve(sizeof(int) * nhist);
        o[i][5] = carve(sizeof(int) * scan_seg_ints((long long)nhist));
    }
    void* base = nullptr;
    if (int rc = stream_scratch(s, off, &base)) return rc;
    char* b = static_cast<char*>(base);
    for (int i = 0; i < count; ++i) {
        GroupJob& j = jobs.job[i];
        auto words = [&](int a) { return reinterpret_cast<unsigned*>(b + o[i][a]); };
        j.k0 = words(0); j.k1 = words(1); j.v0 = words(2); j.v1 = words(3);
        j.hist = reinterpret_cast<int*>(b + o[i][4]);
        j.seg = reinterpret_cast<int*>(b + o[i][5]);
    }
    for (int shift = 0; shift < bits; shift += digit) {
        const bool first = shift == 0;
        const int rc = digit == 8 ? radix_pass<8>(count, jobs, first, n, rows, shift, s)
                     : digit == 10 ? radix_pass<10>(count, jobs, first, n, rows, shift, s) : radix_pass<11>(count, jobs, first, n, rows, shift, s);
        if (rc) return rc;
        for (int i = 0; i < count; ++i) {
            GroupJob& j = jobs.job[i];
            unsigned* t = j.k0; j.k0 = j.k1; j.k1 = t;
            t = j.v0; j.v0 = j.v1; j.v1 = t;
        }
    }
    const dim3 grid((unsigned)((n + kBlock - 1) / kBlock), count);
    if (average) {
        hipLaunchKernelGGL(row_ptr_from_sorted_kernel, grid, dim3(kBlock), 0, s, jobs, n, rows);
        hipLaunchKernelGGL(fill_grouped_kernel<true>, grid, dim3(kBlock), 0, s, jobs, n, rows);
    } else {
        hipLaunchKernelGGL(fill_grouped_kernel<false>, grid, dim3(kBlock), 0, s, jobs, n, rows);
    }
    GNNHIP_LAUNCH_CHECK("csr_group_pairs");
    return GNNHIP_OK;
}

// One grouping, in one launch where that fits.
int csr_group(int rows, long long n, const int* key, int key_stride, const int* payload, int payload_stride, const float* val_in, int average,
              int* row_ptr, int* col_idx, float* val, hipStream_t s)
{
    if (csr_group_small(rows, n, key, key_stride, payload, payload_stride, val_in, average, row_ptr, col_idx, val, nullptr, nullptr, nullptr, s))
        return last_launch_status("csr_group_small");
    GroupJobs jobs{};
    jobs.job[0] = GroupJob{key, payload, val_in, key_stride, payload_stride, row_ptr, col_idx, val};
    return csr_group_pairs(1, jobs, rows, n, average, s);
}

}  // namespace gnnhip

using namespace gnnhip;

extern "C" {

int gnnhip_csr_group_i32(int rows, int n, const int* key, int key_stride, const int* payload, int payload_stride,
                         int average, int* row_ptr, int* col_idx, float* val, void* stream)
{
    GNNHIP_REQUIRE(rows >= 0 && n >= 0 && key_stride >= 1 && payload_stride >= 1, "bad shape in csr_group (rows=%d n=%d)", rows, n);
    GNNHIP_REQUIRE(row_ptr != nullptr, "null row_ptr in csr_group");
    GNNHIP_REQUIRE(n == 0 || (key && payload && col_idx && val), "null array in csr_group");
    GNNHIP_REQUIRE(n == 0 || rows >= 1, "pairs but no rows in csr_group");
    if (int rc = require_ready()) return rc;
    return csr_group(rows, n, key, key_stride, payload, payload_stride, nullptr, average, row_ptr, col_idx, val, as_stream(stream));
}

int gnnhip_csr_group_one_launch(int rows, int n)
{
    SmallLayout lay;
    return small_layout(rows, n, &lay) ? 1 : 0;
}

int gnnhip_csr_consecutive_rows_f32(int rows, const int* row_ptr, int average, int* col_idx, float* val, void* stream)
{
    GNNHIP_REQUIRE(rows >= 0, "negative row count in csr_consecutive_rows");
    if (rows == 0) return GNNHIP_OK;
    GNNHIP_REQUIRE(row_ptr && col_idx && val, "null array in csr_consecutive_rows");
    if (int rc = require_ready()) return rc;
    const unsigned grid = (unsigned)(((long long)rows * kWave + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(consecutive_rows_kernel, dim3(grid), dim3(kBlock), 0, as_stream(stream), rows, row_ptr, average, col_idx, val,
                       static_cast<int*>(nullptr));
    GNNHIP_LAUNCH_CHECK("consecutive_rows");
    return GNNHIP_OK;
}

int gnnhip_csr_consecutive_rows_host_f32(int rows, const int* offsets_host, int average, int* row_ptr, int* col_idx, float* val, void* stream)
{
    GNNHIP_REQUIRE(rows >= 0, "negative row count in csr_consecutive_rows_host");
    GNNHIP_REQUIRE(offsets_host && row_ptr, "null row pointers in csr_consecutive_rows_host");
    GNNHIP_REQUIRE(offsets_host[rows] == 0 || (col_idx && val), "null array in csr_consecutive_rows_host");
    if (int rc = require_ready()) return rc;
    hipStream_t s = as_stream(stream);
    const void* pinned = nullptr;
    if (rows > 0 && offsets_host[rows] > 0)
        if (int rc = stage_in_pinned(s, offsets_host, sizeof(int) * ((size_t)rows + 1), &pinned)) return rc;
    if (!pinned) {
        if (int rc = gnnhip_memcpy_h2d(row_ptr, offsets_host, sizeof(int) * ((size_t)rows + 1), stream)) return rc;
        return (rows > 0 && offsets_host[rows] > 0) ? gnnhip_csr_consecutive_rows_f32(rows, row_ptr, average, col_idx, val, stream) : GNNHIP_OK;
    }
    const unsigned grid = (unsigned)(((long long)rows * kWave + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(consecutive_rows_kernel, dim3(grid), dim3(kBlock), 0, s, rows, static_cast<const int*>(pinned), average, col_idx, val,
                       row_ptr);
    GNNHIP_LAUNCH_CHECK("consecutive_rows");
    return GNNHIP_OK;
}

int gnnhip_csr_group_both_i32(int rows, int n, const int* x, int x_stride, const int* y, int y_stride,
                              int* row_ptr, int* col_idx, float* val, int* t_row_ptr, int* t_col_idx, float* t_val, void* stream)
{
    GNNHIP_REQUIRE(rows >= 0 && n >= 0 && x_stride >= 1 && y_stride >= 1, "bad shape in csr_group_both (rows=%d n=%d)", rows, n);
    GNNHIP_REQUIRE(row_ptr && t_row_ptr, "null row pointers in csr_group_both");
    GNNHIP_REQUIRE(n == 0 || (x && y && col_idx && val && t_col_idx && t_val), "null array in csr_group_both");
    GNNHIP_REQUIRE(n == 0 || rows >= 1, "pairs but no rows in csr_group_both");
    if (int rc = require_ready()) return rc;
    hipStream_t s = as_stream(stream);
    if (csr_group_small(rows, n, y, y_stride, x, x_stride, nullptr, 0, row_ptr, col_idx, val, t_row_ptr, t_col_idx, t_val, s))
        return last_launch_status("csr_group_small");
    GroupJobs jobs{};
    jobs.job[0] = GroupJob{y, x, nullptr, y_stride, x_stride, row_ptr, col_idx, val};
    jobs.job[1] = GroupJob{x, y, nullptr, x_stride, y_stride, t_row_ptr, t_col_idx, t_val};
    return csr_group_pairs(2, jobs, rows, n, 0, s);
}

int gnnhip_csr_transpose_f32(int m, int k, int nnz, const int* row_ptr, const int* col_idx, const float* val,
                             int* t_row_ptr, int* t_col_idx, float* t_val, void* stream)
{
    GNNHIP_REQUIRE(m >= 0 && k >= 0 && nnz >= 0, "bad shape in csr_transpose (m=%d k=%d nnz=%d)", m, k, nnz);
    GNNHIP_REQUIRE(row_ptr && t_row_ptr, "null row pointers in csr_transpose");
    GNNHIP_REQUIRE(nnz == 0 || (col_idx && val && t_col_idx && t_val), "null array in csr_transpose");
    GNNHIP_REQUIRE(nnz == 0 || k >= 1, "entries but no columns in csr_transpose");
    if (int rc = require_ready()) return rc;
    hipStream_t s = as_stream(stream);
    int* row_of = nullptr;
    if (nnz > 0) {
        // the row index of every entry lives in plan scratch (slot 1); the sort itself uses slot 0
        void* p = nullptr;
        if (int rc = stream_scratch_slot(s, 1, sizeof(int) * (size_t)nnz, &p)) return rc;
        row_of = static_cast<int*>(p);
        const unsigned grid = (unsigned)(((long long)m * kWave + kBlock - 1) / kBlock);
        if (m > 0) hipLaunchKernelGGL(expand_rows_kernel, dim3(grid), dim3(kBlock), 0, s, m, row_ptr, row_of);
    }
    return csr_group(k, nnz, col_idx, 1, row_of, 1, val, 0, t_row_ptr, t_col_idx, t_val, s);
}

}  // extern "C"
