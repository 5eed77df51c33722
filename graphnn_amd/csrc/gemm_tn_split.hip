// C = alpha * A^T * B + beta * C for an output of up to 256 x 256 over a very long k: the weight gradients of the
// mean-field levels and of the input stage, dW = [h_0 .. h_{L-1}]^T [u_1 .. u_L] with k = levels x nodes and
// dW_n2l = X^T dmsg with k = nodes (MatMul::Backward, src/nn/matmul.cpp:35-76: x^T * dy through DTensor<GPU>::MM,
// src/tensor/gpu_dense_tensor.cu:192-224).
//
// One workgroup of eight wavefronts holds the whole output in registers and walks one contiguous range of k, so every row
// of A and B is read from memory once per launch (64 x 64 tiles read them up to four times).  The products are formed on
// the bf16 matrix cores from three pieces per operand (bf16_split.h).  An operand is split on its way into LDS: a thread
// takes eight rows of one column, which is one lane's share of v_mfma_f32_32x32x16_bf16, and writes each piece as one
// 128-bit word; words of neighbouring columns lie side by side, so neither the writes nor the reads conflict.  A stage's
// pieces go to the other half of the LDS while the one before is multiplied, and the loads of the one after it are issued
// as soon as that has freed their registers, ahead of the barrier (one per stage).  The workgroups' raw sums go to scratch and
// are added in range order.  Bound by those loads: 300,000 rows, 64 x 64 outputs 36 us (4.2 TB/s), 128 x 128 80 (3.8),
// 256 x 256 245 (2.5: 32 KB on their way per compute unit, which has no registers for more).
#include "bf16_split.h"
#include "buffer_addr.h"

namespace gnnhip {

// gemm.hip
void launch_splitk_reduce(int m, int n, int splits, float alpha, const float* partial, float beta, float* C, int ldc, hipStream_t s);

namespace {

typedef float mfma_f16 __attribute__((ext_vector_type(16)));   // accumulator of a 32 x 32 tile

__device__ __forceinline__ mfma_f16 mfma_32(const bf16_words4& a, const bf16_words4& b, const mfma_f16& c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

constexpr int kTnWaves = 8;
constexpr int kTnBlock = kTnWaves * kWave;

// Operand tiles of MT columns of A and NT columns of B (columns past m / n are zeros); the wavefronts form WR x WC parts
// of the output, KW times over different 16-row groups of a stage of 16 KB rows of k.
template <int MT_, int NT_, int WR_, int WC_, int KW_, int KB_> struct TnShape {
    static constexpr int MT = MT_, NT = NT_, WR = WR_, WC = WC_, KW = KW_, KB = KB_;
    static constexpr int TR = MT / 32 / WR, TC = NT / 32 / WC;           // 32 x 32 tiles of a wavefront
    static constexpr int COLS = MT + NT;
    static constexpr int CHUNKS = COLS / kWave * 2 * KB;                 // 64 columns x 8 rows, the load of one wavefront
    static constexpr int UNITS = (CHUNKS + kTnWaves - 1) / kTnWaves;     // of those per wavefront and stage
    static constexpr int PIECE = 2 * KB * COLS;                          // 128-bit words of one piece of a stage
    static constexpr size_t LDS = 2 * 3 * (size_t)PIECE * 16;
    static constexpr int PER_CU = LDS <= 80 * 1024 ? 2 : 1;              // workgroups that share a compute unit
    static_assert(WR * WC * KW == kTnWaves && KB % KW == 0 && TR >= 1 && TC >= 1, "shape");
};

// TRANSPOSED: the sums are stored [n][m]
template <class S, bool TRANSPOSED>
__global__ __launch_bounds__(kTnBlock, S::PER_CU * kTnWaves / 4) void sgemm_tn_split_kernel(int m, int n, int k, int k_chunk, const float* __restrict__ A, int lda,
                                                                  const float* __restrict__ B, int ldb, float* __restrict__ partial)
{
    extern __shared__ bf16_words4 words[];                // [2 stages][3 pieces][2 KB groups of eight rows][COLS]
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wr = wave % S::WR, wc = wave / S::WR % S::WC, kw = wave / (S::WR * S::WC);
    const long long k_lo = (long long)blockIdx.x * k_chunk;
    const int rows = (int)min((long long)k_chunk, (long long)k - k_lo);      // > 0: the grid covers k exactly
    // this workgroup's rows only: what lies past them reads as zero
    const rsrc_t a_rsrc = make_rsrc(A + (size_t)k_lo * lda, (unsigned)(((size_t)(rows - 1) * lda + m) * 4));
    const rsrc_t b_rsrc = make_rsrc(B + (size_t)k_lo * ldb, (unsigned)(((size_t)(rows - 1) * ldb + n) * 4));

    mfma_f16 acc[S::TR][S::TC];
    // lane l ends with column l % 32 of a tile (of its transpose) and rows 8 (r / 4) + 4 (l / 32) + r % 4
    auto tile_x = [&]() { return lane & 31; };
    auto tile_y = [&](int r) { return 8 * (r / 4) + 4 * (lane >> 5) + r % 4; };

    // A wavefront's share of a stage: UNITS times 64 columns x 8 rows, a column per lane
    float f[S::UNITS][8];
    auto fetch = [&](int r0) {
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) {
            const int chunk = wave + u * kTnWaves;
            if (S::CHUNKS % kTnWaves && chunk >= S::CHUNKS) break;
            const int group = chunk / (S::COLS / kWave), c0 = chunk % (S::COLS / kWave) * kWave;
            const bool is_a = c0 < S::MT;
            const int col = is_a ? c0 + lane : c0 - S::MT + lane;
            const int ld = is_a ? lda : ldb;
            const rsrc_t rsrc = is_a ? a_rsrc : b_rsrc;
            const int voff = col < (is_a ? m : n) ? col * 4 : kBufPastEnd;
#pragma unroll
            for (int i = 0; i < 8; ++i) f[u][i] = buf_load_f(rsrc, voff, (r0 + 8 * group + i) * ld * 4);
        }
    };
    // The scale of the pieces (bf16_split.h) is a column's, for all rows of the workgroup: up at first, and if a large element
    // turned up in some column, everything once more with those columns scaled down.
    __shared__ unsigned char large_in[S::COLS];           // per column
    float largest[S::UNITS];                              // of what this lane has parked
    bool down[S::UNITS];                                  // whether its column is scaled down the second time
    auto park = [&](int buf, unsigned sign, auto again) __attribute__((always_inline)) {
        constexpr bool kAgain = decltype(again)::value;
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) {
            const int chunk = wave + u * kTnWaves;
            if (S::CHUNKS % kTnWaves && chunk >= S::CHUNKS) break;
            const unsigned flip = chunk % (S::COLS / kWave) < S::MT / kWave ? sign : 0u;
            const bool scaled_down = kAgain && down[u];
            const float scale = scaled_down ? kSplitDown : kSplitUp;
            bf16_words4 w[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = f[u][2 * i], y = f[u][2 * i + 1];
                unsigned p[3];
                if (!kAgain) largest[u] = split_max(largest[u], x, y);
                bf16_split2(x * scale, y * scale, scaled_down, p);
                w[0][i] = p[0] ^ flip; w[1][i] = p[1] ^ flip; w[2][i] = p[2] ^ flip;
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) words[(buf * 3 + j) * S::PIECE + chunk * kWave + lane] = w[j];
        }
    };

    // The six products of 16 rows are summed on their own, corrections first, and that sum is added to the running one by the
    // vector unit: one rounding to nearest per 16 rows instead of six by the matrix instruction, which rounds towards minus
    // infinity.  What is left of that drift, one rounding of a 16-row sum, has the opposite sign in every other stage, and in
    // every other workgroup: the pieces of A are negated there, and the sum is subtracted.
    // rms error against float64, relative to the sum of the terms' magnitudes, 128 x 128 over 20,000 rows, A past a ReLU: all
    // products into the running sum 3.3e-9, so 0.9e-9 (general kernel on the FP32 matrix cores 2.6e-9).
    auto run = [&](auto again) __attribute__((always_inline)) {
        constexpr bool kAgain = decltype(again)::value;
        // From four tiles on the pieces of the next stage are formed between the products of the last three tiles; with fewer
        // there is not enough to hide them behind, and the loads would have less time (256 x 256 over 1.5M rows: 1,179 us
        // with the pieces behind the products, 1,130 so).
        constexpr bool kEarly = S::TR * S::TC >= 4;
#pragma unroll
        for (int i = 0; i < S::TR; ++i)
#pragma unroll
            for (int j = 0; j < S::TC; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
        unsigned sign = blockIdx.x & 1 ? 0x80008000u : 0u;    // of the stage being multiplied
        fetch(0);
        park(0, sign, again);
        fetch(16 * S::KB);
        __syncthreads();
        int buf = 0;
        for (int r0 = 0; r0 < rows; r0 += 16 * S::KB) {
            const bool more = r0 + 16 * S::KB < rows;
            const float factor = sign ? -kSplitUpBack * kSplitUpBack : kSplitUpBack * kSplitUpBack;
#pragma unroll
            for (int kb = 0; kb < S::KB / S::KW; ++kb) {
                const bf16_words4* src = words + buf * 3 * S::PIECE + (2 * (kb * S::KW + kw) + (lane >> 5)) * S::COLS + (lane & 31);
                auto load_a = [&](int i, bf16_words4 (&a)[3]) {
#pragma unroll
                    for (int p = 0; p < 3; ++p) a[p] = src[p * S::PIECE + (wr * S::TR + i) * 32];
                };
                bf16_words4 a[S::TR][3], b[3];
#pragma unroll
                for (int i = 0; i < S::TR; ++i) load_a(i, a[i]);
                // Tile after tile, two sums in turn: one is added to the running sum while the products of the other are formed.
                mfma_f16 sum[2];
#pragma unroll
                for (int q = 0; q <= S::TR * S::TC; ++q) {
                    if (kEarly && kb == S::KB / S::KW - 1 && q == S::TR * S::TC - 3) {
                        park(buf ^ 1, sign ^ 0x80008000u, again);
                        fetch(r0 + 2 * 16 * S::KB);
                    }
                    if (q < S::TR * S::TC) {
                        const int i = q % S::TR, j = q / S::TR;
                        if (i == 0) {
#pragma unroll
                            for (int p = 0; p < 3; ++p) b[p] = src[p * S::PIECE + S::MT + (wc * S::TC + j) * 32];
                        }
#pragma unroll
                        for (int r = 0; r < 16; ++r) sum[q & 1][r] = 0.f;
#pragma unroll
                        for (int p = 2; p >= 0; --p)
#pragma unroll
                            for (int o = 2 - p; o >= 0; --o)
                                sum[q & 1] = TRANSPOSED ? mfma_32(b[p], a[i][o], sum[q & 1]) : mfma_32(a[i][o], b[p], sum[q & 1]);
                    }
                    if (q > 0) {
                        const int i = (q - 1) % S::TR, j = (q - 1) / S::TR;
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            float back = factor;
                            if (kAgain) {
                                const int a_col = (wr * S::TR + i) * 32 + (TRANSPOSED ? tile_x() : tile_y(r));
                                const int b_col = (wc * S::TC + j) * 32 + (TRANSPOSED ? tile_y(r) : tile_x());
                                back = (sign ? -1.f : 1.f) * (large_in[a_col] ? kSplitDownBack : kSplitUpBack) *
                                       (large_in[S::MT + b_col] ? kSplitDownBack : kSplitUpBack);
                            }
                            acc[i][j][r] = fmaf(sum[(q - 1) & 1][r], back, acc[i][j][r]);
                        }
                        // here, and not, as the compiler would have it, those of all tiles behind the last product: that many
                        // sums do not fit the registers
                        asm volatile("" : "+v"(acc[i][j]));
                    }
                    if (!kAgain && q > 0 && q < S::TR * S::TC) {
                        // a product, three additions; towards the end the pieces of the next stage as well
                        if (kEarly && kb == S::KB / S::KW - 1 && q >= S::TR * S::TC - 3) {
#pragma unroll
                            for (int x = 0; x < 6; ++x) { __builtin_amdgcn_sched_group_barrier(0x8, 1, 0); __builtin_amdgcn_sched_group_barrier(0x2, 12, 0); }
                        } else {
#pragma unroll
                            for (int x = 0; x < 6; ++x) { __builtin_amdgcn_sched_group_barrier(0x8, 1, 0); __builtin_amdgcn_sched_group_barrier(0x2, 3, 0); }
                        }
                    }
                }
            }
            sign ^= 0x80008000u;
            if (!kEarly && more) {
                park(buf ^ 1, sign, again);
                fetch(r0 + 2 * 16 * S::KB);
            }
            __syncthreads();
            buf ^= 1;
        }
    };
    bool any_large = false;
#pragma unroll
    for (int u = 0; u < S::UNITS; ++u) largest[u] = 0.f;
    run(std::false_type());
#pragma unroll
    for (int u = 0; u < S::UNITS; ++u) any_large |= largest[u] >= kSplitLarge;
    if (__syncthreads_or(any_large)) {                    // the same for all wavefronts
        auto column = [&](int u) { return (wave + u * kTnWaves) % (S::COLS / kWave) * kWave + lane; };
        for (int i = threadIdx.x; i < S::COLS; i += kTnBlock) large_in[i] = 0;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) if (largest[u] >= kSplitLarge) large_in[column(u)] = 1;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) down[u] = large_in[column(u)] != 0;
        run(std::true_type());
    }

    float* part = partial + ((size_t)blockIdx.x * S::KW + kw) * m * n;
#pragma unroll
    for (int i = 0; i < S::TR; ++i)
#pragma unroll
        for (int j = 0; j < S::TC; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = (wr * S::TR + i) * 32 + (TRANSPOSED ? tile_x() : tile_y(r)), col = (wc * S::TC + j) * 32 + (TRANSPOSED ? tile_y(r) : tile_x());
                if (row < m && col < n) part[TRANSPOSED ? (size_t)col * m + row : (size_t)row * n + col] = acc[i][j][r];
            }
}

// From this many multiply-adds on, and over at least so many rows.  Below, the general kernel's ranges of k fill the chip as
// well, and a batch of products runs there in one pair of launches (64 x 64 over 30,000 rows: 18 us there, 14 us here).
constexpr long long kTnMinWork = 1ll << 28, kTnMinK = 8192;

template <class S, bool TRANSPOSED>
int launch_tn_split(int m, int n, int k, float alpha, const float* A, int lda, const float* B, int ldb, float beta, float* C, int ldc,
                    hipStream_t s)
{
    // As many workgroups as the LDS lets run together, each a contiguous range of k of whole stages; not so many that
    // their sums would be more to write and read than the operands.
    const long long want = (long long)kNumCU * S::PER_CU, stage = 16 * S::KB;
    long long chunk = (k + want - 1) / want;
    if (chunk < 4 * stage) chunk = 4 * stage;
    if (chunk < m * n / (m + n)) chunk = m * n / (m + n);
    chunk = (chunk + stage - 1) / stage * stage;
    const int blocks = (int)((k + chunk - 1) / chunk);
    // 32-bit byte offsets inside a workgroup's rows
    const long long ld = lda > ldb ? lda : ldb;
    if ((chunk + 2 * stage) * ld * 4 >= (1ll << 31)) return GNNHIP_EUNSUPPORTED;
    void* q = nullptr;
    if (int rc = stream_scratch_slot(s, 2, sizeof(float) * (size_t)blocks * S::KW * m * n, &q)) return rc;
    float* partial = static_cast<float*>(q);
    static LdsLimit lds_limit;
    GNNHIP_HIP(lds_limit.raise(reinterpret_cast<const void*>(&sgemm_tn_split_kernel<S, TRANSPOSED>), S::LDS));
    hipLaunchKernelGGL((sgemm_tn_split_kernel<S, TRANSPOSED>), dim3((unsigned)blocks), dim3(kTnBlock), S::LDS, s, m, n, k, (int)chunk, A, lda,
                       B, ldb, partial);
    GNNHIP_LAUNCH_CHECK("sgemm_tn_split");
    launch_splitk_reduce(TRANSPOSED ? n : m, TRANSPOSED ? m : n, blocks * S::KW, alpha, partial, beta, C, ldc, s);
    GNNHIP_LAUNCH_CHECK("sgemm_tn_split sums");
    return GNNHIP_OK;
}

// m <= n
template <bool TRANSPOSED>
int choose_tn_split(int m, int n, int k, float alpha, const float* A, int lda, const float* B, int ldb, float beta, float* C, int ldc,
                    hipStream_t s)
{
#define GNNHIP_TN(...) return launch_tn_split<TnShape<__VA_ARGS__>, TRANSPOSED>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s)
    if (n <= 64) GNNHIP_TN(64, 64, 2, 2, 2, 2);
    if (n <= 128) {
        if (m <= 64) GNNHIP_TN(64, 128, 2, 2, 2, 2);
        GNNHIP_TN(128, 128, 2, 4, 1, 1);
    }
    if (m <= 64) GNNHIP_TN(64, 256, 1, 8, 1, 1);
    // one workgroup per compute unit: in the 128 registers that two would leave a lane, the sums in turn are spilled (1.5M rows: 792 us, 675 so)
    if (m <= 128) GNNHIP_TN(128, 256, 2, 4, 1, 2);
    GNNHIP_TN(256, 256, 4, 2, 1, 1);
#undef GNNHIP_TN
}

}  // namespace

// GNNHIP_EUNSUPPORTED (nothing launched): the product keeps the general kernel.  The batch of weight gradients asks here
// too, so that a product gets the bits it has when done alone.
int gemm_tn_split_dispatch(int m, int n, int k, float alpha, const float* A, int lda, const float* B, int ldb, float beta, float* C,
                           int ldc, hipStream_t s)
{
    if (m < 1 || n < 1 || m > 256 || n > 256 || k < kTnMinK || (long long)m * n * k < kTnMinWork) return GNNHIP_EUNSUPPORTED;
    if (m <= n) return choose_tn_split<false>(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
    // the narrower operand first
    return choose_tn_split<true>(n, m, k, alpha, B, ldb, A, lda, beta, C, ldc, s);
}

}  // namespace gnnhip
