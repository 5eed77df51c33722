// Runs of consecutive graphs of at most `cap` nodes together ("bins"): block-diagonal graphs like any other, which a
// workgroup of a forward kernel carries as one.
//
// Every 64 consecutive graphs (a segment) are packed on their
// own by one wavefront (first fit in batch order; a bin never crosses such a boundary, which costs about one
// partly filled bin per segment): a ballot per bin gives a 64-bit word in which the graphs that open one are set, and the lanes
// of those graphs write the segment's records, from record 64 x segment on.  The forward kernel finds bin b by a prefix sum over the set
// bits of the words, one of them per lane, so the segments need not know of each other: a wavefront each and three trips to
// memory, 4.7 us for 3,001 graphs.  (One workgroup that packed the whole batch, to number the bins itself, took 8.5.  Without
// this launch, a workgroup of the forward kernel either packs all segments, which costs it more than this launch from
// some 500 bins on, or numbers bins by its own segment, which spreads them unevenly over the dies: 1,500 graphs at hidden 64 72
// us where bins numbered through the batch take 45.)  A graph of more than cap nodes is a bin of its own (the forward kernel
// refuses it).  Output: words[segment], then one record of kOrderRec ints per bin: first graph, first node, nodes, first entry, end of
// entries, graphs.
#ifndef GNNHIP_GRAPH_BINS_H
#define GNNHIP_GRAPH_BINS_H

#include "gnnhip_internal.h"

namespace gnnhip {

// CHECKED: nothing is known about s_row_ptr.  A segment whose graphs are no ascending ranges of nodes, of at most `limit` nodes each (at least cap), that
// begin at node 0 and end at node N, gets the word 0 (a segment that is packed opens at least one bin), and *refused is set to 0 for the forward
// kernel to set when it comes upon such a word.
struct BinsArgs {
    int B, cap;
    const int *a_row_ptr, *s_row_ptr;
    int* bins;
    int N, limit;
    int* refused;
};

namespace {

constexpr int kOrderRec = 8;                     // ints per record (32-byte records)
constexpr int kBinBlock = 128;
// ints ahead of the records: the words of the segments, in whole records
__host__ __device__ inline size_t bin_words_ints(int B) { return ((size_t)((B + kWave - 1) / kWave) * 2 + kOrderRec - 1) / kOrderRec * kOrderRec; }
// and all of them
__host__ __device__ inline size_t bin_ints(int B) { return bin_words_ints(B) + kOrderRec * (size_t)((B + kWave - 1) / kWave * kWave); }

// one segment, by one wavefront
template <bool CHECKED>
__device__ __forceinline__ void pack_segment(int seg, const BinsArgs& a)
{
    const int B = a.B, cap = a.cap, N = a.N, limit = a.limit;
    const int* __restrict__ a_row_ptr = a.a_row_ptr;
    const int* __restrict__ s_row_ptr = a.s_row_ptr;
    int* __restrict__ bins = a.bins;
    const int lane = threadIdx.x & (kWave - 1);
    const int nlive = min(kWave, B - seg * kWave);
    if (nlive <= 0) return;
    int start = 0, end = 0;                      // first node and end of the lane's graph
    if (lane < nlive) { start = s_row_ptr[seg * kWave + lane]; end = s_row_ptr[seg * kWave + lane + 1]; }
    if constexpr (CHECKED) {
        if (seg == 0 && lane == 0) *a.refused = 0;
        const int g = seg * kWave + lane;
        const bool bad = start < 0 || end < start || end > N || end - start > limit || (g == 0 && start != 0) || (g == B - 1 && end != N);
        if (__any(lane < nlive && bad)) {
            if (lane == 0) reinterpret_cast<unsigned long long*>(bins)[seg] = 0;
            return;
        }
    }
    unsigned long long opens = 0;
    int first = 0;
    while (first < nlive) {
        const int node0 = __builtin_amdgcn_readlane(start, first);
        opens |= 1ull << first;
        // lanes from `first` on whose graph no longer fits behind node0: the bin ends before the first of them
        const unsigned long long stop = __ballot(lane >= first && (lane >= nlive || end - node0 > cap));
        int next = stop ? (int)__builtin_ctzll(stop) : kWave;
        if (next == first) next = first + 1;                         // larger than cap: alone
        first = __builtin_amdgcn_readfirstlane(next);
    }
    if (lane == 0) reinterpret_cast<unsigned long long*>(bins)[seg] = opens;
    // a lane whose graph opens a bin writes its record (a bin the forward kernel will refuse gets no entry range)
    const unsigned long long behind = lane == kWave - 1 ? 0 : opens >> (lane + 1);
    const int ng = (behind ? lane + 1 + (int)__builtin_ctzll(behind) : nlive) - lane;
    const int n = __shfl(end, min(max(lane + ng - 1, 0), kWave - 1), kWave) - start;
    if (!((opens >> lane) & 1ull)) return;
    int e0 = 0, e1 = 0;
    if (n >= 0 && n <= (CHECKED ? limit : cap)) { e0 = a_row_ptr[start]; e1 = a_row_ptr[start + n]; }
    int* rec = bins + bin_words_ints(B) + (size_t)(seg * kWave + __popcll(opens & ((1ull << lane) - 1ull))) * kOrderRec;
    *reinterpret_cast<int4*>(rec) = make_int4(seg * kWave + lane, start, n, e0);
    *reinterpret_cast<int2*>(rec + 4) = make_int2(e1, ng);
}

template <bool CHECKED>
__global__ __launch_bounds__(kBinBlock) void graph_bins_kernel(BinsArgs a)
{
    pack_segment<CHECKED>(__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kBinBlock / kWave) + threadIdx.x / kWave)), a);
}

// Where the record of a bin is.  A wavefront asks for its bins in ascending order and goes on
// from the words that held the last one (from the first word for every bin: 500,000 graphs of 1 to 3 nodes, hidden 16 950 us, 709 so;
// 60,000 145, 141).
struct BinFinder {
    int nseg, seg = 0, before = 0;               // 64 words from seg on, bins of the words before them
    const unsigned long long* words;
    __device__ BinFinder(int B, const int* bins) : nseg((B + kWave - 1) / kWave), words(reinterpret_cast<const unsigned long long*>(bins)) {}
    // the place of the record of a bin, or -1 past the last one
    __device__ __forceinline__ int find(int bin)
    {
        const int lane = threadIdx.x & (kWave - 1);
        for (; seg < nseg; seg += kWave) {
            const int count = seg + lane < nseg ? __popcll(words[seg + lane]) : 0;
            const int through = before + wave_inclusive_scan_i(count);
            const unsigned long long behind = __ballot(bin < through);
            if (behind) {
                const int at = (int)__builtin_ctzll(behind);
                return (seg + at) * kWave + bin - __builtin_amdgcn_readlane(through - count, at);
            }
            before = __builtin_amdgcn_readlane(through, kWave - 1);
        }
        return -1;
    }
};

}  // namespace
}  // namespace gnnhip

#endif
