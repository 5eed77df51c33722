// The wide mean-field level (C = 128 or 256) with its contraction on the bf16 matrix cores:
//     h_out = ReLU((A * h_in) * W + msg)
// (examples/graph_classification/src/kernel_mean_field.cpp:35-42), every product formed from three bf16 pieces of
// either operand (bf16_split.h: fp32 sums of exact products), and the backward pass of a level through the same
// machinery.
//
// On FP32 matrix cores the contraction takes 8,192 cycles of a SIMD per 16 rows at C = 256, twice what the level's HBM
// traffic takes; six bf16 products take 3,072.  The structure is that of
// level_wide.hip: a persistent workgroup of eight wavefronts per compute unit, W in registers for the whole launch,
// the rows of a pass summed into one LDS tile while the matrix cores read the other, one batch of six row loads per
// 16-row block.  What is different:
//   * A row is split into its pieces once, by the wavefront that summed it, and lies in LDS as three bf16 planes, its scale
//     (bf16_split.h) behind them; a column of W has a scale of its own.
//   * W in pieces takes 192 of a lane's 256 registers at C = 256.  The few fragments that do not fit are read from LDS;
//     spilled to scratch memory they were reloaded behind the gather's loads, in whose order they had to wait (1.45 times the
//     launch).
//   * A wavefront whose rows hold more entries than the tops of the remaining blocks can take starts a second batch in
//     the middle of a block; gathering behind the pass would hold up the other seven.
//
// 299,536 nodes, 659,010 entries, C = 256, first level apart: 380 (FP32 matrix cores) -> 276 us per level (0.93 GB of
// activations at 3.4 TB/s), backward 474 -> 428 us (1.85 GB at 4.3 TB/s).  Counted there: 0.64 GB fetched and 0.31 GB written, matrix
// pipes busy 40 % of the cycles, 3.8 other instructions per matrix instruction of 16 cycles (1.9 of them vector ones, which
// split the rows, 1.5 scalar ones, which steer the gather), no bank conflicts: neither memory nor the matrix pipes, but two
// wavefronts per SIMD, too few to issue past each other's waits, that meet at the barrier of every pass.  Summing the
// corrections apart from the large products costs 5 % of the launch (265 -> 277) and takes the rms error from 2.2 .. 3.1e-8 of
// the terms' sum to 1e-8 (FP32 matrix cores: 2.4 .. 2.8e-8).
//
// Used by the inference forward and by the backward pass.  The levels of a training forward stay on level_wide.hip:
// the sign of its outputs decides which gradients pass, so two roundings of the same sum give gradients that differ
// by whole terms wherever a pre-activation is within rounding of zero (a few of 400 million per iteration).
#include "bf16_split.h"
#include "level_wide.h"

namespace gnnhip {
namespace {

// C = 256: W in pieces takes 192 of a lane's 256 registers, and what does not fit would be reloaded from scratch memory
// right behind the gather's loads, in whose order it would have to wait.  The third piece of this many contraction steps
// of the first column block is read from LDS instead (one 128-bit read per step).
template <int C, int TR, bool BWD> constexpr int wide_lds_fragments() { return C != 256 ? 0 : TR == 16 ? (BWD ? 8 : 11) : (BWD ? 7 : 6); }

// Everything that steers the gather (row pointers, column indices, edge weights) is uniform
// across the wavefront and is fetched with scalar loads: the values land in scalar registers, cost
// no vector instruction to broadcast, and are counted apart from vector memory operations, so
// waiting for them never waits for a store.
// RELU_IN: the gathered rows count as ReLU(row) (the first level reading msg where h0 was not stored)
// TR: rows per pass (16 or 32)
// BWD: the backward pass of a level through the same machinery.  The CSR arrays are those of A^T, h_in is dz, the
//      summed rows u = A^T dz are also stored to u_out as each one is finished (they are the other factor of the
//      weight gradient), the contraction takes W transposed (g = u W^T), and the epilogue, instead of adding msg and
//      applying ReLU, lets g through where the rows of `msg` (here: the embedding whose ReLU the gradient passes next,
//      or null for no gate) are positive and adds what it stores to acc_io (or null).
template <int C, int WAVES, bool RELU_IN, int TR, bool BWD = false>
__global__ __launch_bounds__(WAVES * kWave) void s2v_level_split_kernel(
    int N, int tiles_per_block, const int* __restrict__ row_ptr, const int* __restrict__ col_idx,
    const float* __restrict__ val, const float* __restrict__ h_in, const float* __restrict__ W,
    const float* __restrict__ msg, float* __restrict__ h_out, float* __restrict__ u_out, float* __restrict__ acc_io)
{
    constexpr int KS = C / 32;                   // contraction steps
    constexpr int CW = C / WAVES;                // output columns per wavefront
    constexpr int NB = CW / 16;                  // 16-column blocks per wavefront
    constexpr int VEC = C / kWave;               // gathered floats per lane
    // A tile in LDS is [3 pieces][2 halves of the columns][kTileRows][LDT] of bf16, with room behind every half row (the first
    // piece's first half keeps the row's scale there).  A 128-bit LDS read serves sixteen lanes per
    // cycle, lanes 0-3, 12-15 of one sixteen together with lanes 4-11 of its neighbour; rows that start in distinct
    // 16-byte bank groups and neighbours that read the two halves (a multiple of 256 bytes apart) make that free of conflicts.
    constexpr int LDT = C / 2 + 8;
    constexpr int kTileRows = TR;
    constexpr int RPW = kTileRows / WAVES;       // rows gathered per wavefront per pass
    constexpr int kHalf = kTileRows * LDT;
    constexpr int kPiece = 2 * kHalf;            // one piece of every element of a tile
    static_assert(kHalf * 2 % 256 == 0, "halves start at the same bank");
    constexpr int NF = wide_lds_fragments<C, TR, BWD>();
    using vec_t = typename VecT<VEC>::type;

    extern __shared__ unsigned short tiles[];    // two tiles [3 pieces][kTileRows][LDT] of bf16: one read by the matrix
                                                 // cores, the other being filled for the next pass
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int col0 = wave * CW;
    const int gather_off = (lane >> 5) * kHalf + (wave * RPW) * LDT + (lane & 31) * VEC;
    const int k_lane = (q & 1) * (C / 2) + (q >> 1) * 8;            // contraction step s of this lane: k = k_lane + 16 s .. + 7

    // The matrix instruction rounds its sum towards minus infinity.  The middle half of the contraction steps is formed with
    // -W on the negated sum, so that the drift of one half of the steps cancels that of the other.
    auto negated = [](int s) { return s >= KS / 4 && s < KS - KS / 4; };

    // W^T operand, in pieces: wreg[jb][s] holds W[k_lane + 16 s + 0..7][col0 + 16 jb + t]; BWD: of W itself,
    // W[col0 + 16 jb + t][k_lane + 16 s + 0..7] (buffer loads: one lane offset, the steps as scalar offsets, so no 64-bit
    // address per element is formed)
    bf16_words4 wreg[NB][KS][3];
    float* w_down = reinterpret_cast<float*>(tiles + 2 * 3 * kPiece);         // [C]: a column's scale up over its scale
    bf16_words4* w_lds = reinterpret_cast<bf16_words4*>(w_down + C) + (size_t)wave * NF * kWave + lane;
    bool any_down;                               // columns of this wavefront that are scaled down (bf16_split.h): uniform
    {
        const rsrc_t w_rsrc = make_rsrc(W, (unsigned)(C * C * 4));
        const int w_lane_off = BWD ? ((col0 + t) * C + k_lane) * 4 : (k_lane * C + col0 + t) * 4;
        unsigned long long large[NB];            // lanes that hold a large weight
        auto load_w = [&](auto again) {
            constexpr bool kAgain = decltype(again)::value;
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                float largest = 0.f;
                const bool scaled_down = kAgain && ((large[jb] >> t) & 0x0001000100010001ull);      // in any quarter of the column
                const float scale = scaled_down ? kSplitDown : kSplitUp;
                if (kAgain && q == 0) w_down[col0 + 16 * jb + t] = scaled_down ? kSplitUp / kSplitDown : 1.f;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    float w[8];
                    if constexpr (BWD) {         // consecutive floats of one row of W
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const float4 v = buf_load4(w_rsrc, w_lane_off + 16 * C * 4 * jb, s * 64 + 16 * h);
                            w[4 * h + 0] = v.x; w[4 * h + 1] = v.y; w[4 * h + 2] = v.z; w[4 * h + 3] = v.w;
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i) w[i] = buf_load_f(w_rsrc, w_lane_off + 64 * jb, (16 * s + i) * (C * 4));
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (!kAgain) largest = split_max(largest, w[2 * i], w[2 * i + 1]);
                        unsigned p[3];
                        bf16_split2(w[2 * i] * scale, w[2 * i + 1] * scale, scaled_down, p);
                        wreg[jb][s][0][i] = p[0]; wreg[jb][s][1][i] = p[1]; wreg[jb][s][2][i] = p[2];
                    }
                    if (negated(s)) {
#pragma unroll
                        for (int p = 0; p < 3; ++p) wreg[jb][s][p] ^= 0x80008000u;
                    }
                    if (jb * KS + s < NF) w_lds[(jb * KS + s) * kWave] = wreg[jb][s][2];
                }
                if (!kAgain) large[jb] = __ballot(largest >= kSplitLarge);
            }
        };
        load_w(std::false_type());
        unsigned long long all = 0;
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) all |= large[jb];
        any_down = all != 0;
        if (any_down) load_w(std::true_type());                  // again, with the columns of large weights scaled down
    }

    const int ntiles = (int)(((long long)N + kTileRows - 1) / kTileRows);
    const int tile_begin = (int)min((long long)blockIdx.x * tiles_per_block, (long long)ntiles);
    const int tile_end = (int)min((long long)ntiles, (long long)tile_begin + tiles_per_block);
    if (tile_begin >= tile_end) return;

    // ---- loaders.  The RPW + 1 row pointers of a pass sit in lanes 0..RPW of one vector register; columns
    //      and weights of a batch are uniform and come through scalar loads (weights as bit patterns
    //      so that selecting them stays on the scalar unit).
    auto load_rowptrs = [&](int tile_id) {
        const long long r0 = (long long)tile_id * kTileRows + wave * RPW;
        int v = 0;
        if (lane <= RPW) v = row_ptr[min(r0 + lane, (long long)N)];
        return v;
    };
    const int* val_bits = reinterpret_cast<const int*>(val);
    // entries [s, s + kInFlight) of the CSR arrays.  What lies past the end of the wavefront's rows is
    // loaded but never added, so the batch is read as it lies.  Only a batch that would run past the end
    // of the arrays starts earlier; batch_ready() then shifts it into place.  The entry count that bounds
    // these reads is the matrix's own (row_ptr[N], read here), never a count passed by the host.  A matrix
    // with fewer entries than one batch is read entry by entry, with zeros behind the last one.
    const int nnz = row_ptr[N];
    auto load_batch = [&](const int* arr, int s, Batch& b) {
        if (nnz < kInFlight) {
            batch_load_short(b, arr, nnz);
            return s;
        }
        const int base = max(min(s, nnz - kInFlight), 0);
        batch_load(b, arr + base);
        return s - base;                         // by how many entries the batch has to be shifted
    };
    auto batch_ready = [&](Batch& b, int shift) {
        batch_wait(b);
        for (; shift > 0; --shift) {             // only at the very end of the arrays
            b.lo.x = b.lo.y; b.lo.y = b.lo.z; b.lo.z = b.lo.w; b.lo.w = b.hi.x; b.hi.x = b.hi.y;
        }
    };
    const rsrc_t h_rsrc = make_rsrc(h_in, (unsigned)((size_t)N * C * 4));
    auto issue = [&](const Batch& c, vec_t (&x)[kInFlight]) {
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
            x[u] = BufLoad<VEC>::get(h_rsrc, lane * (VEC * 4), batch_get(c, u) * (C * 4));     // N C 4 < 2^32 (host-checked)
    };

    // ---- state of the gather of one pass: entries [e, ee) of the wavefront's RPW rows, taken in order;
    //      a row goes to LDS when its last entry has been added
    int e = 0, ee = 0, lr = 0, row_end = 0, rpv = 0;
    unsigned short* dstp = nullptr;
    float acc[VEC];
    rsrc_t u_rsrc = make_rsrc(u_out, 0);         // BWD: the rows of u_out that the pass being gathered covers
    auto begin = [&](int rp_lanes, int eb, int eend, unsigned short* dst, int tile_id) {
        rpv = rp_lanes;
        e = eb; ee = eend; lr = 0;
        row_end = __builtin_amdgcn_readlane(rpv, 1);
        dstp = dst;
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
        if constexpr (BWD) {
            const long long r0 = (long long)tile_id * kTileRows;
            const long long rows = max(min((long long)N - r0, (long long)kTileRows), 0ll);      // none past the last pass
            u_rsrc = make_rsrc(u_out + (size_t)min(r0, (long long)N) * C, (unsigned)(rows * (C * 4)));
        }
    };
    auto flush_row = [&]() {
        unsigned p[VEC / 2][3];
        float largest = 0.f;
#pragma unroll
        for (int i = 0; i < VEC; i += 2) largest = split_max(largest, acc[i], acc[i + 1]);
        const bool scaled_down = __any(largest >= kSplitLarge);
        if (scaled_down) {
#pragma unroll
            for (int i = 0; i < VEC / 2; ++i) bf16_split2(acc[2 * i] * kSplitDown, acc[2 * i + 1] * kSplitDown, true, p[i]);
        } else {
#pragma unroll
            for (int i = 0; i < VEC / 2; ++i) bf16_split2(acc[2 * i] * kSplitUp, acc[2 * i + 1] * kSplitUp, false, p[i]);
        }
        // behind the row's first half: what undoes its scale
        if (lane == 31) *reinterpret_cast<float*>(dstp + VEC) = scaled_down ? kSplitDownBack : kSplitUpBack;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if constexpr (VEC == 4) *reinterpret_cast<uint2*>(dstp + j * kPiece) = make_uint2(p[0][j], p[1][j]);
            else *reinterpret_cast<unsigned*>(dstp + j * kPiece) = p[0][j];
        }
        if constexpr (BWD)                        // rows past N lie outside the descriptor
            BufStore<VEC>::put(u_rsrc, lane * (VEC * 4), (wave * RPW + lr) * (C * 4), *reinterpret_cast<vec_t*>(acc));
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
        dstp += LDT;
        ++lr;
        row_end = __builtin_amdgcn_readlane(rpv, min(lr + 1, RPW));
    };
    auto consume = [&](const Batch& a, const vec_t (&x)[kInFlight]) {
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            if (e + u < ee) {
                while (e + u >= row_end) flush_row();          // rows ending here (possibly empty ones)
                vec_fma<VEC, RELU_IN>(acc, __int_as_float(batch_get(a, u)), x[u]);
            }
        }
        e += kInFlight;
    };
    auto finish = [&]() { while (lr < RPW) flush_row(); };      // the open row and empty rows after it

    // Output of the last finished 16-row block, stored at the top of the following block (or at the end
    // of the pass): a store then has a whole contraction between its issue and the next wait on
    // vector memory.  msg and h_out are addressed through descriptors that cover the rows of the
    // current pass only, so rows past N fall outside and need no predicate.
    float4 outv[NB];
    int out_rt = -1;                             // block of this pass held in outv, -1: none
#pragma unroll
    for (int jb = 0; jb < NB; ++jb) outv[jb] = f4_zero();
    const int lane_off = (t * C + col0 + 4 * q) * 4;              // byte offset of this lane inside a 16-row block
    rsrc_t msg_rsrc = make_rsrc(msg, 0), out_rsrc = make_rsrc(h_out, 0), acc_rsrc = make_rsrc(acc_io, 0);
    auto store_pending = [&]() {
        if (out_rt >= 0) {
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) buf_store4(out_rsrc, lane_off + out_rt * (16 * C * 4) + 64 * jb, 0, outv[jb]);
        }
        out_rt = -1;
    };

    Batch cC, aC;                                // columns / weights of the next batch to issue / to sum
    cC.lo = i32x4{0, 0, 0, 0}; cC.hi = i32x2{0, 0};
    aC.lo = i32x4{0, 0, 0, 0}; aC.hi = i32x2{0, 0};
    int cShift = 0, aShift = 0;                  // shifts owed to cC / aC when they are next read

    // ---- first pass: its gather has nothing to hide behind
    int rp_next = load_rowptrs(tile_begin);      // row pointers of the next pass to gather
    int ebN = __builtin_amdgcn_readlane(rp_next, 0), eeN = __builtin_amdgcn_readlane(rp_next, RPW);
    begin(rp_next, ebN, eeN, tiles + gather_off, tile_begin);
    while (e < ee) {
        vec_t x[kInFlight];
        cShift = load_batch(col_idx, e, cC);
        aShift = load_batch(val_bits, e, aC);
        batch_ready(cC, cShift);
        batch_ready(aC, aShift);
        issue(cC, x);
        consume(aC, x);
    }
    finish();
    ebN = eeN = 0;
    if (tile_begin + 1 < tile_end) {
        rp_next = load_rowptrs(tile_begin + 1);
        ebN = __builtin_amdgcn_readlane(rp_next, 0);
        eeN = __builtin_amdgcn_readlane(rp_next, RPW);
        if (ebN < eeN) { cShift = load_batch(col_idx, ebN, cC); aShift = load_batch(val_bits, ebN, aC); }
    }
    __syncthreads();

    for (int tile_id = tile_begin; tile_id < tile_end; ++tile_id) {
        const long long row0 = (long long)tile_id * kTileRows;
        const int parity = (tile_id - tile_begin) & 1;
        const unsigned short* cur = tiles + parity * (3 * kPiece);
        const bool has_next = tile_id + 1 < tile_end;
        const bool has_next2 = tile_id + 2 < tile_end;
        begin(rp_next, ebN, eeN, tiles + (parity ^ 1) * (3 * kPiece) + gather_off, tile_id + 1);   // empty when !has_next
        {
            const long long left = (long long)N - row0;
            const unsigned bytes = (unsigned)(min(left, (long long)kTileRows) * (C * 4));
            out_rsrc = make_rsrc(h_out + (size_t)row0 * C, bytes);
            msg_rsrc = make_rsrc(msg ? msg + (size_t)row0 * C : nullptr, msg ? bytes : 0u);   // no msg: every load reads 0
            if constexpr (BWD) acc_rsrc = make_rsrc(acc_io ? acc_io + (size_t)row0 * C : nullptr, acc_io ? bytes : 0u);
        }
        if (has_next2) rp_next = load_rowptrs(tile_id + 2);

        // ---- contraction and epilogue, one 16-row block at a time; each block also carries one batch
        //      of the next pass's gather, issued before its matrix instructions and summed after them
#pragma unroll 1
        for (int rt = 0; rt < kTileRows / 16; ++rt) {
            // msg is asked for now and added after the contraction (as the accumulators' initial value it
            // would have to arrive before the first matrix instruction)
            float4 mm[NB], aa[BWD ? NB : 1];
            mfma_f4 acc_m[NB];
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                if constexpr (!BWD) mm[jb] = buf_load4(msg_rsrc, lane_off + rt * (16 * C * 4) + 64 * jb, 0);
                acc_m[jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};
            }
            vec_t x[kInFlight];
            const bool batch = e < ee;
            if (batch) { batch_ready(cC, cShift); issue(cC, x); }
            store_pending();
            // where the follower of this batch starts: inside this pass, or (after the last block) at the
            // first entry of the next pass; its columns travel while the matrix cores work
            int ns = 0, nend = 0;
            if (rt < kTileRows / 16 - 1) {
                if (e + kInFlight < ee) { ns = e + kInFlight; nend = ee; }
            } else if (kTileRows > 16 && e + kInFlight >= ee) {
                ns = ebN; nend = eeN;                     // both zero when there is no next pass
            }
            // (a 16-row pass has one block: ebN/eeN still describe the pass being gathered, the row pointers of
            // the one after it arrive during this block, so its first batch is asked for after the block)

            const unsigned short* src = cur + (q & 1) * kHalf + (rt * 16 + t) * LDT + (q >> 1) * 8;
            // Two rounds over the contraction steps: first the five products that are corrections, whose sum is about 2^-8 of
            // the result, then the products of the first pieces.  The result itself is then rounded once per step (KS times)
            // and not six times: rms error against float64, relative to the sum of the terms' magnitudes, 1e-8 where all six
            // in one round leave 2.2e-8 to 3.1e-8 and the FP32 matrix cores 2.4e-8 to 2.8e-8 (one sign: 6e-8 against 1.7e-7),
            // for 5 us more per level (the first pieces of the tile are read twice).  The first round takes the negated
            // steps first, so the sum changes its sign three times.
            auto turn = [&]() {
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) acc_m[jb] = -acc_m[jb];
            };
            auto first_round = [&](int i) { return i < KS / 2 ? i + KS / 4 : i < 3 * KS / 4 ? i - KS / 2 : i; };
            auto piece = [&](int j, int step) { return *reinterpret_cast<const bf16_words4*>(src + j * kPiece + 16 * step); };
            // A piece of the tile operand is read for the next step as soon as this step's products with it are issued, so
            // that each read has six or more matrix instructions to arrive in; the first pieces of the second round's first
            // three steps take the same registers.
            bool again = false;
            const float back = *reinterpret_cast<const float*>(cur + (rt * 16 + t) * LDT + C / 2) * kSplitUpBack;
            bf16_words4 b[3];
#pragma unroll
            for (int j = 2; j >= 0; --j) b[j] = piece(j, first_round(0));
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int f = first_round(s);
                if (s == KS / 2) turn();
                bf16_words4 w3[NB];
#pragma unroll
                for (int jb = 0; jb < NB; ++jb)
                    if (jb * KS + f < NF) w3[jb] = w_lds[(jb * KS + f) * kWave];
#pragma unroll
                for (int j = 2; j >= 0; --j) {
#pragma unroll
                    for (int i = 2 - j; i >= (j == 0 ? 1 : 0); --i)
#pragma unroll
                        for (int jb = 0; jb < NB; ++jb)
                            acc_m[jb] = mfma_bf16(i == 2 && jb * KS + f < NF ? w3[jb] : wreg[jb][f][i], b[j], acc_m[jb]);
                    b[j] = s + 1 < KS ? piece(j, first_round(s + 1)) : piece(0, 2 - j);
                    __builtin_amdgcn_sched_barrier(0);            // keeps the read-ahead where it is written
                }
                // the follower's columns are asked for here, behind the first wait for LDS of this block: a
                // scalar load in flight counts with the LDS reads, and the next wait is 6 NB matrix instructions away
                if (s == 0 && ns < nend) cShift = load_batch(col_idx, ns, cC);
                if (s == KS / 2 - 1 && batch && ee - (e + kInFlight) > kInFlight * (kTileRows / 16 - 1 - rt)) {
                    // more entries than the tops of the blocks that are left can take: this wavefront takes a second batch
                    // in this block (in the open behind the pass it would keep the other seven waiting)
                    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
                    batch_ready(aC, aShift);
                    consume(aC, x);
                    aShift = load_batch(val_bits, e, aC);
                    if (rt == kTileRows / 16 - 1) cShift = load_batch(col_idx, e, cC);
                    batch_ready(cC, cShift);
                    batch_ready(aC, aShift);                  // both have to land before the paths join
                    aShift = 0;
                    issue(cC, x);
                    ns = nend = 0;
                    if (e + kInFlight < ee) {
                        if (rt < kTileRows / 16 - 1) { ns = e + kInFlight; nend = ee; }
                    } else if (kTileRows > 16 && rt == kTileRows / 16 - 1) {
                        ns = ebN; nend = eeN;
                    }
                    again = ns < nend;
                }
                if (s == KS / 2 && again) cShift = load_batch(col_idx, ns, cC);
            }
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                if (s > 0 && negated(s) != negated(s - 1)) turn();
                bf16_words4& a = b[2 - s % 3];
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) acc_m[jb] = mfma_bf16(wreg[jb][s][0], a, acc_m[jb]);
                if (s + 3 < KS) a = piece(0, s + 3);
                __builtin_amdgcn_sched_barrier(0);
            }
            // One unconditional wait for everything this block asked for (gathered rows, msg).  The loads
            // and their uses sit under separate conditions; without this the compiler has to assume a
            // path on which they are still in flight and waits at the top of the next block instead,
            // where the wait also covers the stores issued just before it.
            if constexpr (BWD) {
                // the gate and the old values of acc_io are asked for here, where the operands of the contraction have left
                // their registers, and arrive while the gathered rows are summed; where a buffer is null its loads touch
                // nothing
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) mm[jb] = buf_load4(msg_rsrc, lane_off + rt * (16 * C * 4) + 64 * jb, 0);
#pragma unroll
                for (int jb = 0; jb < NB; ++jb) aa[jb] = buf_load4(acc_rsrc, lane_off + rt * (16 * C * 4) + 64 * jb, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_waitcnt(kWaitVmcnt0 + (BWD ? 2 * NB : 0));
            if (batch) { batch_ready(aC, aShift); consume(aC, x); }
            if (ns < nend) aShift = load_batch(val_bits, ns, aC);
            if (rt == 0) {                                // the row pointers asked for at the top have arrived
                ebN = eeN = 0;
                if (has_next2) {
                    ebN = __builtin_amdgcn_readlane(rp_next, 0);
                    eeN = __builtin_amdgcn_readlane(rp_next, RPW);
                }
            }
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                float4 f = make_float4(back, back, back, back);
                if (any_down) {
                    const float4 d = *reinterpret_cast<const float4*>(w_down + col0 + 16 * jb + 4 * q);
                    f.x *= d.x; f.y *= d.y; f.z *= d.z; f.w *= d.w;
                }
                if constexpr (BWD) {
                    float4 v = make_float4(acc_m[jb][0] * f.x, acc_m[jb][1] * f.y, acc_m[jb][2] * f.z, acc_m[jb][3] * f.w);
                    if (msg) {                   // past the ReLU whose output these rows are
                        v.x = mm[jb].x > 0.f ? v.x : 0.f; v.y = mm[jb].y > 0.f ? v.y : 0.f;
                        v.z = mm[jb].z > 0.f ? v.z : 0.f; v.w = mm[jb].w > 0.f ? v.w : 0.f;
                    }
                    if (acc_io) {                // every row belongs to one pass: nobody else touches it during the launch
                        const float4 a = make_float4(aa[jb].x + v.x, aa[jb].y + v.y, aa[jb].z + v.z, aa[jb].w + v.w);
                        buf_store4(acc_rsrc, lane_off + rt * (16 * C * 4) + 64 * jb, 0, a);
                    }
                    outv[jb] = v;
                } else {
                    const float4 v = make_float4(fmaf(acc_m[jb][0], f.x, mm[jb].x), fmaf(acc_m[jb][1], f.y, mm[jb].y),
                                                 fmaf(acc_m[jb][2], f.z, mm[jb].z), fmaf(acc_m[jb][3], f.w, mm[jb].w));
                    outv[jb] = relu_max4(v);
                }
            }
            out_rt = rt;
        }
        if (kTileRows == 16 || e < ee) {                  // more batches than blocks: finish in the open
            while (e < ee) {
                vec_t x[kInFlight];
                cShift = load_batch(col_idx, e, cC);
                aShift = load_batch(val_bits, e, aC);
                batch_ready(cC, cShift);
                batch_ready(aC, aShift);
                issue(cC, x);
                consume(aC, x);
            }
            if (ebN < eeN) { cShift = load_batch(col_idx, ebN, cC); aShift = load_batch(val_bits, ebN, aC); }
        }
        if (has_next) finish();
        store_pending();
        __syncthreads();                                  // the tile just filled is complete, the other one is free
    }
}

// The same over few rows at C = 256, where the kernel above is its start: a wavefront there splits 32 columns of W (3,300 vector
// instructions) ahead of the first row, and all of a tile's matrix instructions are one compute unit's.  Here a workgroup takes 16 rows, a
// wavefront sums two of them, and the workgroups of the grid's y share the columns: `blocks` wavefronts have 16 of them each, split while
// the entries are on their way.  Row sums, pieces and products have the order of the kernel above, so every bit is its.
// 286 rows 11.5 -> 7.5 us per level of a forward, backward 14.7 -> 8.3; 1,760 rows 12.0 -> 10.0 and 15.4 -> 11.2.  Over more than 2,048 rows a second
// workgroup per compute unit would follow the first.  (Sixteen wavefronts, a row each, leave a lane 128 registers, of which W takes
// 96: spilled, 13 to 32 us.)
constexpr int kFewWaves = 8, kFewEach = 16 / kFewWaves;         // wavefronts, rows that each sums
template <int C, bool RELU_IN, bool BWD>
__global__ __launch_bounds__(kFewWaves * kWave) void s2v_level_split_few_kernel(
    int N, int blocks, const int* __restrict__ row_ptr, const int* __restrict__ col_idx, const float* __restrict__ val,
    const float* __restrict__ h_in, const float* __restrict__ W, const float* __restrict__ msg, float* __restrict__ h_out,
    float* __restrict__ u_out, float* __restrict__ acc_io)
{
    constexpr int KS = C / 32, VEC = C / kWave, LDT = C / 2 + 8, kHalf = 16 * LDT, kPiece = 2 * kHalf, kFlight = 8;
    static_assert(VEC == 4, "a wavefront holds a row as one 128-bit word per lane");
    __shared__ __align__(16) unsigned short tile[3 * kPiece];    // [3 pieces][2 halves of the columns][16][LDT], as above
    __shared__ float w_down[C];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int row0 = blockIdx.x * 16, rows = min(16, N - row0);
    const int col0 = 16 * (blockIdx.y * blocks + wave);
    const bool live = wave < blocks && col0 < C;                 // uniform: this wavefront multiplies
    const int k_lane = (q & 1) * (C / 2) + (q >> 1) * 8;         // contraction step s: k = k_lane + 16 s .. + 7
    auto negated = [](int s) { return s >= KS / 4 && s < KS - KS / 4; };

    // ---- what is asked for first: W, then this wavefront's row pointers and entries
    float w[KS][8];
    if (live) {
        const rsrc_t w_rsrc = make_rsrc(W, (unsigned)(C * C * 4));
        const int w_lane_off = BWD ? ((col0 + t) * C + k_lane) * 4 : (k_lane * C + col0 + t) * 4;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if constexpr (BWD) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 v = buf_load4(w_rsrc, w_lane_off, s * 64 + 16 * h);
                    w[s][4 * h + 0] = v.x; w[s][4 * h + 1] = v.y; w[s][4 * h + 2] = v.z; w[s][4 * h + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) w[s][i] = buf_load_f(w_rsrc, w_lane_off, (16 * s + i) * (C * 4));
            }
        }
    }
    // row 8 r + wave for r = 0, 1: an entry per lane
    int start[kFewEach], end[kFewEach], c_lane[kFewEach];
    float v_lane[kFewEach];
    const rsrc_t h_rsrc = make_rsrc(h_in, (unsigned)N * (C * 4));
#pragma unroll
    for (int r = 0; r < kFewEach; ++r) {
        const int row = min(r * kFewWaves + wave, rows);         // past the last row: no entries
        start[r] = row_ptr[row0 + row];
        end[r] = row_ptr[min(row0 + row + 1, row0 + rows)];
    }
    auto ask_entries = [&](int r, int base) {
        const bool ok = base + lane < end[r];
        c_lane[r] = ok ? col_idx[base + lane] : 0;
        v_lane[r] = ok ? val[base + lane] : 0.f;
    };
#pragma unroll
    for (int r = 0; r < kFewEach; ++r) ask_entries(r, start[r]);

    // ---- W in pieces
    bf16_words4 wreg[KS][3];
    bool any_down = false;
    if (live) {
        float largest = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int i = 0; i < 8; i += 2) largest = split_max(largest, w[s][i], w[s][i + 1]);
        const unsigned long long large = __ballot(largest >= kSplitLarge);
        const bool down = (large >> t) & 0x0001000100010001ull;  // in any quarter of the column
        any_down = large != 0;
        const float scale = down ? kSplitDown : kSplitUp;
        if (q == 0) w_down[col0 + t] = down ? kSplitUp / kSplitDown : 1.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                unsigned p[3];
                bf16_split2(w[s][2 * i] * scale, w[s][2 * i + 1] * scale, down, p);
                const unsigned sign = negated(s) ? 0x80008000u : 0u;
                wreg[s][0][i] = p[0] ^ sign; wreg[s][1][i] = p[1] ^ sign; wreg[s][2][i] = p[2] ^ sign;
            }
        }
    }

    // ---- the rows: the first entries of both, then the rest of each
    float4 x[kFewEach][kFlight];
    auto ask_rows = [&](int r, int e, int count) {
#pragma unroll
        for (int u = 0; u < kFlight; ++u) {
            const int c = __builtin_amdgcn_readlane(c_lane[r], min(e + u, kWave - 1));
            x[r][u] = buf_load4(h_rsrc, e + u < count ? lane * 16 : kBufPastEnd, c * (C * 4));
        }
    };
#pragma unroll
    for (int r = 0; r < kFewEach; ++r) ask_rows(r, 0, min(end[r] - start[r], kWave));
#pragma unroll
    for (int r = 0; r < kFewEach; ++r) {
        float acc[VEC] = {0.f, 0.f, 0.f, 0.f};
        for (int base = start[r]; base < end[r]; base += kWave) {            // uniform
            const int count = min(end[r] - base, kWave);
            if (base > start[r]) { ask_entries(r, base); ask_rows(r, 0, count); }
            for (int e = 0; e < count; e += kFlight) {
                if (e > 0) ask_rows(r, e, count);
#pragma unroll
                for (int u = 0; u < kFlight; ++u) {
                    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v_lane[r]), min(e + u, kWave - 1)));
                    if (e + u < count) vec_fma<VEC, RELU_IN>(acc, a, x[r][u]);
                }
            }
        }
        float largest = 0.f;
#pragma unroll
        for (int i = 0; i < VEC; i += 2) largest = split_max(largest, acc[i], acc[i + 1]);
        const bool down = __any(largest >= kSplitLarge);
        unsigned p[2][3];
        const float scale = down ? kSplitDown : kSplitUp;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (down) bf16_split2(acc[2 * i] * scale, acc[2 * i + 1] * scale, true, p[i]);
            else bf16_split2(acc[2 * i] * scale, acc[2 * i + 1] * scale, false, p[i]);
        }
        const int row = r * kFewWaves + wave;
        unsigned short* dst = tile + (lane >> 5) * kHalf + row * LDT + (lane & 31) * VEC;
        if (lane == 31) *reinterpret_cast<float*>(dst + VEC) = down ? kSplitDownBack : kSplitUpBack;     // behind the row's first half
#pragma unroll
        for (int j = 0; j < 3; ++j) *reinterpret_cast<uint2*>(dst + j * kPiece) = make_uint2(p[0][j], p[1][j]);
        if constexpr (BWD) {
            if (row < rows && blockIdx.y == 0)
                *reinterpret_cast<float4*>(u_out + (size_t)(row0 + row) * C + lane * 4) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        }
    }
    // what the epilogue reads: columns col0 + 4 q .. + 3 of row t (rows past N lie outside the descriptors)
    const int off = ((row0 + t) * C + col0 + 4 * q) * 4;
    const rsrc_t msg_rsrc = make_rsrc(msg, msg ? (unsigned)N * (C * 4) : 0u);
    const rsrc_t acc_rsrc = make_rsrc(acc_io, BWD && acc_io ? (unsigned)N * (C * 4) : 0u);
    float4 mm = f4_zero(), aa = f4_zero();
    if (live) {
        mm = buf_load4(msg_rsrc, off, 0);
        if constexpr (BWD) aa = buf_load4(acc_rsrc, off, 0);
    }
    __syncthreads();
    if (!live) return;                           // no barrier follows

    // ---- products: the corrections first, negated steps ahead of the others, then those of the first pieces
    const unsigned short* src = tile + (q & 1) * kHalf + t * LDT + (q >> 1) * 8;
    auto piece = [&](int j, int step) { return *reinterpret_cast<const bf16_words4*>(src + j * kPiece + 16 * step); };
    const float back = *reinterpret_cast<const float*>(tile + t * LDT + C / 2) * kSplitUpBack;
    auto first_round = [&](int i) { return i < KS / 2 ? i + KS / 4 : i < 3 * KS / 4 ? i - KS / 2 : i; };
    mfma_f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KS; ++i) {
        const int s = first_round(i);
        if (i == KS / 2) sum = -sum;
#pragma unroll
        for (int j = 2; j >= 0; --j) {
            const bf16_words4 b = piece(j, s);
#pragma unroll
            for (int k = 2 - j; k >= (j == 0 ? 1 : 0); --k) sum = mfma_bf16(wreg[s][k], b, sum);
        }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        if (s > 0 && negated(s) != negated(s - 1)) sum = -sum;
        sum = mfma_bf16(wreg[s][0], piece(0, s), sum);
    }
    float4 f = make_float4(back, back, back, back);
    if (any_down) {
        const float4 d = *reinterpret_cast<const float4*>(w_down + col0 + 4 * q);
        f.x *= d.x; f.y *= d.y; f.z *= d.z; f.w *= d.w;
    }
    if (t >= rows) return;
    float* out = h_out + (size_t)(row0 + t) * C + col0 + 4 * q;
    if constexpr (BWD) {
        float4 v = make_float4(sum[0] * f.x, sum[1] * f.y, sum[2] * f.z, sum[3] * f.w);
        if (msg) {
            v.x = mm.x > 0.f ? v.x : 0.f; v.y = mm.y > 0.f ? v.y : 0.f;
            v.z = mm.z > 0.f ? v.z : 0.f; v.w = mm.w > 0.f ? v.w : 0.f;
        }
        if (acc_io)
            *reinterpret_cast<float4*>(acc_io + (size_t)(row0 + t) * C + col0 + 4 * q) = make_float4(aa.x + v.x, aa.y + v.y, aa.z + v.z, aa.w + v.w);
        *reinterpret_cast<float4*>(out) = v;
    } else {
        const float4 v = make_float4(fmaf(sum[0], f.x, mm.x), fmaf(sum[1], f.y, mm.y), fmaf(sum[2], f.z, mm.z), fmaf(sum[3], f.w, mm.w));
        *reinterpret_cast<float4*>(out) = relu_max4(v);
    }
}

template <int C, bool RELU_IN, bool BWD>
int launch_level_split_few(int N, const int* row_ptr, const int* col_idx, const float* val, const float* h_in, const float* W,
                           const float* msg, float* h_out, hipStream_t s, float* u_out = nullptr, float* acc_io = nullptr)
{
    const int tiles = (N + 15) / 16;
    int share = C / 64;                          // four blocks of columns to a workgroup as long as there are compute units for it
    while (share > 2 && share * tiles > kNumCU) share /= 2;              // a workgroup has eight wavefronts
    hipLaunchKernelGGL((s2v_level_split_few_kernel<C, RELU_IN, BWD>), dim3(tiles, share), dim3(kFewWaves * kWave), 0, s, N, C / 16 / share, row_ptr, col_idx,
                       val, h_in, W, msg, h_out, u_out, acc_io);
    GNNHIP_LAUNCH_CHECK(BWD ? "s2v_level_split_few backward" : "s2v_level_split_few");
    return GNNHIP_OK;
}

template <int C, int WAVES, bool RELU_IN, int TR, bool BWD = false>
int launch_level_split_t(int N, const int* row_ptr, const int* col_idx, const float* val, const float* h_in,
                      const float* W, const float* msg, float* h_out, hipStream_t s, float* u_out = nullptr, float* acc_io = nullptr)
{
    if ((unsigned long long)N * C * 4ull >= (1ull << 32)) return GNNHIP_EUNSUPPORTED;   // 32-bit buffer offsets
    constexpr int kTileRows = TR;
    const long long ntiles = ((long long)N + kTileRows - 1) / kTileRows;
    // workgroups that fit one compute unit together: two at C = 128 (107 registers per lane, 55 KB of LDS each)
    constexpr int kPerCU = (C == 128) ? 2 : 1;
    const long long slots = (long long)kNumCU * kPerCU;
    const long long per = (ntiles + slots - 1) / slots;              // contiguous run of tiles per workgroup
    const long long blocks = (ntiles + per - 1) / per;
    const size_t smem = 2 * 3 * 2 * sizeof(unsigned short) * kTileRows * (C / 2 + 8) + sizeof(float) * C +
                        sizeof(bf16_words4) * (size_t)wide_lds_fragments<C, TR, BWD>() * WAVES * kWave;
    static LdsLimit lds_limit;                                       // one per kernel instantiation
    GNNHIP_HIP(lds_limit.raise(reinterpret_cast<const void*>(&s2v_level_split_kernel<C, WAVES, RELU_IN, TR, BWD>), smem));
    hipLaunchKernelGGL((s2v_level_split_kernel<C, WAVES, RELU_IN, TR, BWD>), dim3((unsigned)blocks), dim3(WAVES * kWave), smem, s,
                       N, (int)per, row_ptr, col_idx, val, h_in, W, msg, h_out, u_out, acc_io);
    GNNHIP_LAUNCH_CHECK(BWD ? "s2v_level_split backward" : "s2v_level_split");
    return GNNHIP_OK;
}

// Rows per pass: 32 (two tiles of 64 rows do not fit the LDS at C = 256), 16 on matrices with fewer 32-row passes than
// twice the workgroups.
template <int C, int WAVES, bool RELU_IN>
int launch_level_split(int N, const int* row_ptr, const int* col_idx, const float* val, const float* h_in,
                      const float* W, const float* msg, float* h_out, hipStream_t s)
{
    constexpr int kSlots = kNumCU * ((C == 128) ? 2 : 1);
    if (N >= 2 * kSlots * 32) return launch_level_split_t<C, WAVES, RELU_IN, 32>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s);
    return launch_level_split_t<C, WAVES, RELU_IN, 16>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s);
}

// The backward pass: same choice of rows per pass.
template <int C, int WAVES>
int launch_level_split_backward(int N, const int* row_ptr, const int* col_idx, const float* val, const float* dz, const float* W,
                               float* u, float* g_prev, const float* gate, float* acc, hipStream_t s)
{
    constexpr int kSlots = kNumCU * ((C == 128) ? 2 : 1);
    if (N >= 2 * kSlots * 32) return launch_level_split_t<C, WAVES, false, 32, true>(N, row_ptr, col_idx, val, dz, W, gate, g_prev, s, u, acc);
    return launch_level_split_t<C, WAVES, false, 16, true>(N, row_ptr, col_idx, val, dz, W, gate, g_prev, s, u, acc);
}

}  // namespace

int level_split_dispatch(int N, int C, const int* row_ptr, const int* col_idx, const float* val,
                        const float* h_in, const float* W, const float* msg, float* h_out, bool relu_in, hipStream_t s)
{
    switch (C) {
    case 128:
        return relu_in ? launch_level_split<128, 8, true>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s)
                       : launch_level_split<128, 8, false>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s);
    case 256:
        if (N <= kFewRows / 2)
            return relu_in ? launch_level_split_few<256, true, false>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s)
                           : launch_level_split_few<256, false, false>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s);
        return relu_in ? launch_level_split<256, 8, true>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s)
                       : launch_level_split<256, 8, false>(N, row_ptr, col_idx, val, h_in, W, msg, h_out, s);
    }
    return GNNHIP_EUNSUPPORTED;
}

// u = A' dz (stored) and g_prev = u W^T past the gate of `gate` (may be null), added to acc (may be null): the wide
// kernel's backward variant over the CSR arrays of A' = A^T.
int level_split_backward_dispatch(int N, int C, const int* row_ptr, const int* col_idx, const float* val, const float* dz, const float* W,
                                 float* u, float* g_prev, const float* gate, float* acc, hipStream_t s)
{
    switch (C) {
    case 128: return launch_level_split_backward<128, 8>(N, row_ptr, col_idx, val, dz, W, u, g_prev, gate, acc, s);
    case 256:
        if (N <= kFewRows / 2) return launch_level_split_few<256, false, true>(N, row_ptr, col_idx, val, dz, W, gate, g_prev, s, u, acc);
        return launch_level_split_backward<256, 8>(N, row_ptr, col_idx, val, dz, W, u, g_prev, gate, acc, s);
    }
    return GNNHIP_EUNSUPPORTED;
}

}  // namespace gnnhip
