// Fused mean-field level for wide hidden sizes (C = 128 or 256):
//     h_out = ReLU((A * h_in) * W + bias + msg)
// the operator chain MatMul(sparse) -> MatMul -> ElewiseAdd -> ReLU of
// examples/graph_classification/src/kernel_mean_field.cpp:35-42 in one launch.
//
// At C = 256 the C x C contraction is 2 N C^2 = 131 kflop per node against
// 3 KB of activation traffic per node: on FP32 matrix cores (157 TFLOP/s) the
// contraction takes about twice as long as the HBM traffic, so this kernel is
// organised around keeping the matrix pipes fed.
//
// This kernel forms the levels of a training forward (and the level entries); level_wide_split.hip does inference and
// the backward pass on the bf16 matrix cores and says why the two are kept apart.
//
// One persistent workgroup of 8 wavefronts per compute unit.  W never moves
// after start-up: wavefront w keeps the W^T operand of its C/8 output columns
// in registers (C = 256: 128 registers per lane, half of the register file of
// the compute unit across the 8 wavefronts).  Per pass over TR rows (64; 32 or 16
// on matrices too small to give every compute unit two 64-row passes):
//   1. gather-sum  wavefront w sums the neighbour rows of TR/8 rows, the whole
//                  wavefront across the C columns of a row, six row loads in
//                  flight, and parks the sums in an LDS tile [TR][C+4];
//   2. contraction v_mfma_f32_16x16x4_f32, out^T = W^T * tile^T: the lane
//                  (q = lane/16, t = lane%16) feeds k = (C/4) q + s at step s, so
//                  four steps of its tile operand are one 128-bit LDS read, and it
//                  ends up owning row t, four consecutive columns per block;
//   3. epilogue    + bias + msg, ReLU, 128-bit stores (issued at the top of the
//                  next 16-row block).
// The tile is double-buffered and the gather of pass p+1 is spread, one batch
// of six row loads per 16-row block, over the contraction of pass p; the CSR
// indices are fetched one batch (columns, weights) or one pass (row pointers)
// further ahead still.  Only a wavefront whose rows hold more than six entries
// per 16-row block of the pass (24 at TR = 64) gathers in the open.
//
// What shaped the code (measured on MI355X):
//   * While a wavefront streams FP32 matrix instructions, every other
//     instruction issued on that SIMD, by either wavefront and of any kind
//     (vector, scalar, LDS, memory), gets about one issue slot per matrix
//     instruction (14 ns) instead of one per 2 ns.  The budget is therefore one
//     non-matrix instruction per matrix instruction; beyond it the matrix pipe
//     idles.  Hence: CSR indices through scalar loads (no broadcast
//     instructions), buffer addressing (a gathered row costs one scalar shift
//     and one load; rows past N are dropped by the descriptor's size, not by a
//     predicate), msg/bias added after the contraction in 8 + 8 adds.
//   * Vector memory operations retire in order, so any wait for a load also
//     waits for every store issued before it.  Stores are therefore issued
//     right before a contraction, never right before a wait.
//   * The loads of a batch and their uses sit under separate (uniform)
//     conditions; the compiler then assumes a path on which loads are still in
//     flight and waits at the top of the next block.  One explicit wait after
//     the contraction removes that.
#include "level_wide.h"

// Phase accounting for a timing build of this file; expands to nothing in the library.
#ifndef GNNHIP_PHASE_ACC
#define GNNHIP_PHASE_ACC(i)
#define GNNHIP_PHASE_INIT
#define GNNHIP_PHASE_FINI
#endif


namespace gnnhip {
namespace {

// Everything that steers the gather (row pointers, column indices, edge weights) is uniform
// across the wavefront and is fetched with scalar loads: the values land in scalar registers, cost
// no vector instruction to broadcast, and are counted apart from vector memory operations, so
// waiting for them never waits for a store.  That matters because on this hardware the FP32 matrix
// instructions and ordinary vector instructions do not overlap: every vector instruction issued by
// either wavefront of a SIMD takes time away from its matrix pipe.
// RELU_IN: the gathered rows count as ReLU(row) (the first level reading msg where h0 was not stored)
// TR: rows per pass (16, 32 or 64)
template <int C, int WAVES, bool RELU_IN, int TR>
__global__ __launch_bounds__(WAVES * kWave) void s2v_level_wide_kernel(
    int N, int tiles_per_block, const int* __restrict__ row_ptr, const int* __restrict__ col_idx,
    const float* __restrict__ val, const float* __restrict__ h_in, const float* __restrict__ W,
    const float* __restrict__ msg, const float* __restrict__ bias, float* __restrict__ h_out)
{
    constexpr int KS = C / 4;                    // contraction steps
    constexpr int kWideBlock = WAVES * kWave;
    constexpr int CW = C / WAVES;                // output columns per wavefront
    constexpr int NB = CW / 16;                  // 16-column blocks per wavefront
    constexpr int VEC = C / kWave;               // gathered floats per lane
    constexpr int LDT = C + 4;                   // LDS row stride: rows 0..7 start in distinct 16-byte bank groups
    constexpr int kTileRows = TR;
    constexpr int RPW = kTileRows / WAVES;       // rows gathered per wavefront per pass
    using vec_t = typename VecT<VEC>::type;

    extern __shared__ float tiles[];             // two tiles [kTileRows][LDT]: one read by the matrix cores,
                                                 // the other being filled for the next pass
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int col0 = wave * CW;
    const int gather_off = (wave * RPW) * LDT + lane * VEC;
    float* bias_lds = tiles + 2 * kTileRows * LDT;      // [C], read in the epilogue without a trip to memory
    if (bias)
        for (int i = threadIdx.x; i < C; i += kWideBlock) bias_lds[i] = bias[i];

    // W^T operand: wreg[jb][s] = W[KS q + s][col0 + 16 jb + t]
    // (buffer loads: one lane offset, the steps as scalar offsets, so no 64-bit address per element is formed)
    float wreg[NB][KS];
    {
        const rsrc_t w_rsrc = make_rsrc(W, (unsigned)(C * C * 4));
        const int w_lane_off = ((KS * q) * C + col0 + t) * 4;
#pragma unroll
        for (int jb = 0; jb < NB; ++jb)
#pragma unroll
            for (int s = 0; s < KS; ++s)
                wreg[jb][s] = buf_load_f(w_rsrc, w_lane_off + 64 * jb, s * (C * 4));
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
    float* dstp = nullptr;
    float acc[VEC];
    auto begin = [&](int rp_lanes, int eb, int eend, float* dst) {
        rpv = rp_lanes;
        e = eb; ee = eend; lr = 0;
        row_end = __builtin_amdgcn_readlane(rpv, 1);
        dstp = dst;
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    };
    auto flush_row = [&]() {
        *reinterpret_cast<vec_t*>(dstp) = *reinterpret_cast<vec_t*>(acc);
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
    rsrc_t msg_rsrc = make_rsrc(msg, 0), out_rsrc = make_rsrc(h_out, 0);
    auto store_pending = [&]() {
        if (out_rt >= 0) {
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) buf_store4(out_rsrc, lane_off + out_rt * (16 * C * 4) + 64 * jb, 0, outv[jb]);
        }
        out_rt = -1;
    };

    GNNHIP_PHASE_INIT
    Batch cC, aC;                                // columns / weights of the next batch to issue / to sum
    cC.lo = i32x4{0, 0, 0, 0}; cC.hi = i32x2{0, 0};
    aC.lo = i32x4{0, 0, 0, 0}; aC.hi = i32x2{0, 0};
    int cShift = 0, aShift = 0;                  // shifts owed to cC / aC when they are next read

    // ---- first pass: its gather has nothing to hide behind
    int rp_next = load_rowptrs(tile_begin);      // row pointers of the next pass to gather
    int ebN = __builtin_amdgcn_readlane(rp_next, 0), eeN = __builtin_amdgcn_readlane(rp_next, RPW);
    begin(rp_next, ebN, eeN, tiles + gather_off);
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
    GNNHIP_PHASE_ACC(0);

    for (int tile_id = tile_begin; tile_id < tile_end; ++tile_id) {
        const long long row0 = (long long)tile_id * kTileRows;
        const int parity = (tile_id - tile_begin) & 1;
        const float* cur = tiles + parity * (kTileRows * LDT);
        const bool has_next = tile_id + 1 < tile_end;
        const bool has_next2 = tile_id + 2 < tile_end;
        begin(rp_next, ebN, eeN, tiles + (parity ^ 1) * (kTileRows * LDT) + gather_off);   // empty when !has_next
        {
            const long long left = (long long)N - row0;
            const unsigned bytes = (unsigned)(min(left, (long long)kTileRows) * (C * 4));
            out_rsrc = make_rsrc(h_out + (size_t)row0 * C, bytes);
            msg_rsrc = make_rsrc(msg ? msg + (size_t)row0 * C : nullptr, msg ? bytes : 0u);   // no msg: every load reads 0
        }
        if (has_next2) rp_next = load_rowptrs(tile_id + 2);

        // ---- contraction and epilogue, one 16-row block at a time; each block also carries one batch
        //      of the next pass's gather, issued before its matrix instructions and summed after them
#pragma unroll 1
        for (int rt = 0; rt < kTileRows / 16; ++rt) {
            // msg is asked for now and added after the contraction (as the accumulators' initial value it
            // would have to arrive before the first matrix instruction)
            float4 mm[NB];
            mfma_f4 acc_m[NB];
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                mm[jb] = buf_load4(msg_rsrc, lane_off + rt * (16 * C * 4) + 64 * jb, 0);
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
            GNNHIP_PHASE_ACC(1);

            const float* src = cur + (rt * 16 + t) * LDT + KS * q;
            // the tile operand is read two 128-bit words (eight contraction steps) ahead of its use
            float4 b_cur[2], b_nxt[2];
            b_cur[0] = *reinterpret_cast<const float4*>(src);
            b_cur[1] = *reinterpret_cast<const float4*>(src + 4);
#pragma unroll
            for (int s8 = 0; s8 < KS / 8; ++s8) {
                if (s8 + 1 < KS / 8) {
                    b_nxt[0] = *reinterpret_cast<const float4*>(src + 8 * (s8 + 1));
                    b_nxt[1] = *reinterpret_cast<const float4*>(src + 8 * (s8 + 1) + 4);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 b = b_cur[h];
                    const int s0 = 8 * s8 + 4 * h;
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc_m[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][s0 + 0], b.x, acc_m[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc_m[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][s0 + 1], b.y, acc_m[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc_m[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][s0 + 2], b.z, acc_m[jb], 0, 0, 0);
#pragma unroll
                    for (int jb = 0; jb < NB; ++jb) acc_m[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[jb][s0 + 3], b.w, acc_m[jb], 0, 0, 0);
                }
                // the follower's columns are asked for here, behind the first wait for LDS of this block: a
                // scalar load in flight counts with the LDS reads, and the next wait is 16 matrix instructions away
                if (s8 == 0 && ns < nend) cShift = load_batch(col_idx, ns, cC);
                __builtin_amdgcn_sched_barrier(0);            // keeps the read-ahead where it is written
                b_cur[0] = b_nxt[0]; b_cur[1] = b_nxt[1];
            }
            GNNHIP_PHASE_ACC(2);
            // One unconditional wait for everything this block asked for (gathered rows, msg).  The loads
            // and their uses sit under separate conditions; without this the compiler has to assume a
            // path on which they are still in flight and waits at the top of the next block instead,
            // where the wait also covers the stores issued just before it.
            __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
            if (batch) { batch_ready(aC, aShift); consume(aC, x); }
            if (ns < nend) aShift = load_batch(val_bits, ns, aC);
            if (rt == 0) {                                // the row pointers asked for at the top have arrived
                ebN = eeN = 0;
                if (has_next2) {
                    ebN = __builtin_amdgcn_readlane(rp_next, 0);
                    eeN = __builtin_amdgcn_readlane(rp_next, RPW);
                }
            }
            GNNHIP_PHASE_ACC(3);
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                acc_m[jb][0] += mm[jb].x; acc_m[jb][1] += mm[jb].y; acc_m[jb][2] += mm[jb].z; acc_m[jb][3] += mm[jb].w;
            }
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) {
                float4 v = make_float4(acc_m[jb][0], acc_m[jb][1], acc_m[jb][2], acc_m[jb][3]);
                if (bias) {
                    const float4 b4 = *reinterpret_cast<const float4*>(bias_lds + col0 + 16 * jb + 4 * q);
                    v.x += b4.x; v.y += b4.y; v.z += b4.z; v.w += b4.w;
                }
                outv[jb] = make_float4(relu_ref(v.x), relu_ref(v.y), relu_ref(v.z), relu_ref(v.w));
            }
            out_rt = rt;
            GNNHIP_PHASE_ACC(4);
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
        GNNHIP_PHASE_ACC(5);
        __syncthreads();                                  // the tile just filled is complete, the other one is free
        GNNHIP_PHASE_ACC(6);
    }
    GNNHIP_PHASE_FINI
}

template <int C, int WAVES, bool RELU_IN, int TR>
int launch_level_wide_t(int N, const int* row_ptr, const int* col_idx, const float* val, const float* h_in,
                      const float* W, const float* msg, const float* bias, float* h_out, hipStream_t s)
{
    if ((unsigned long long)N * C * 4ull >= (1ull << 32)) return GNNHIP_EUNSUPPORTED;   // 32-bit buffer offsets
    constexpr int kTileRows = TR;
    const long long ntiles = ((long long)N + kTileRows - 1) / kTileRows;
    // workgroups that fit one compute unit together: two at C = 128 (82 registers per lane, 68 KB of LDS each)
    constexpr int kPerCU = (C == 128) ? 2 : 1;
    const long long slots = (long long)kNumCU * kPerCU;
    const long long per = (ntiles + slots - 1) / slots;              // contiguous run of tiles per workgroup
    const long long blocks = (ntiles + per - 1) / per;
    const size_t smem = sizeof(float) * (2 * kTileRows * (C + 4) + C);
    static LdsLimit lds_limit;                                       // one per kernel instantiation
    GNNHIP_HIP(lds_limit.raise(reinterpret_cast<const void*>(&s2v_level_wide_kernel<C, WAVES, RELU_IN, TR>), smem));
    hipLaunchKernelGGL((s2v_level_wide_kernel<C, WAVES, RELU_IN, TR>), dim3((unsigned)blocks), dim3(WAVES * kWave), smem, s,
                       N, (int)per, row_ptr, col_idx, val, h_in, W, msg, bias, h_out);
    GNNHIP_LAUNCH_CHECK("s2v_level_wide");
    return GNNHIP_OK;
}

// Rows per pass.  The contraction of a 64-row pass keeps one compute unit's matrix pipes busy for 14 us at
// C = 256, so a matrix with fewer passes than twice the compute units is cut into shorter ones.
template <int C, int WAVES, bool RELU_IN>
int launch_level_wide(int N, const int* row_ptr, const int* col_idx, const float* val, const float* h_in,
                      const float* W, const float* msg, const float* bias, float* h_out, hipStream_t s)
{
    constexpr int kSlots = kNumCU * ((C == 128) ? 2 : 1);
    if (N >= 2 * kSlots * 64) return launch_level_wide_t<C, WAVES, RELU_IN, 64>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s);
    if (N >= 2 * kSlots * 32) return launch_level_wide_t<C, WAVES, RELU_IN, 32>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s);
    return launch_level_wide_t<C, WAVES, RELU_IN, 16>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s);
}

}  // namespace

// Whether N rows of C floats have a wide kernel (32-bit buffer offsets).
bool level_wide_covers(int N, int C)
{
    return (C == 128 || C == 256) && (unsigned long long)N * (unsigned)C * 4ull < (1ull << 32);
}

int level_wide_dispatch(int N, int C, long long nnz, const int* row_ptr, const int* col_idx, const float* val,
                        const float* h_in, const float* W, const float* msg, const float* bias, float* h_out, bool relu_in,
                        hipStream_t s)
{
    (void)nnz;                                   // the kernel bounds its index reads with row_ptr[N]
    switch (C) {
    case 128:
        return relu_in ? launch_level_wide<128, 8, true>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s)
                       : launch_level_wide<128, 8, false>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s);
    case 256:
        return relu_in ? launch_level_wide<256, 8, true>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s)
                       : launch_level_wide<256, 8, false>(N, row_ptr, col_idx, val, h_in, W, msg, bias, h_out, s);
    }
    return GNNHIP_EUNSUPPORTED;
}

}  // namespace gnnhip
