// C = alpha * A^T * B + beta * C for an output of up to 256 x 256 over a very long k: the weight gradients of the
// mean-field levels and of the input stage, dW = [h_0 .. h_{L-1}]^T [u_1 .. u_L] with k = levels x nodes and
// dW_n2l = X^T dmsg with k = nodes (MatMul::Backward, src/nn/matmul.cpp:35-76: x^T * dy through DTensor<GPU>::MM,
// src/tensor/gpu_dense_tensor.cu:192-224).
//
// One workgroup of eight wavefronts holds the whole output in registers and walks one contiguous range of k, so every row
// of A and B is read from memory once per launch (64 x 64 tiles read them up to four times).  The products are formed on
// the bf16 matrix cores from three pieces per operand (bf16_split.h).  An operand is split on its way into LDS: a thread
// takes eight rows of one column, which is one lane's share of v_mfma_f32_32x32x16_bf16, and writes each piece as one
// 128-bit word; words of neighbouring columns lie side by side, so neither the writes nor the reads conflict.  While a
// stage is multiplied the next one is on its way from memory, and it goes to the other half of the LDS behind the
// products (one barrier per stage).  The workgroups' raw sums go to scratch and are added in range order.
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
    // four tiles in the 128 registers of two workgroups: one sum of 16 rows at a time, its operand read again from LDS
    static constexpr bool KEEP_A = !(PER_CU == 2 && TR * TC >= 4);
    static constexpr int SUMS = KEEP_A ? TR : 1;
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
#pragma unroll
    for (int i = 0; i < S::TR; ++i)
#pragma unroll
        for (int j = 0; j < S::TC; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

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
    auto park = [&](int buf, unsigned sign) {
#pragma unroll
        for (int u = 0; u < S::UNITS; ++u) {
            const int chunk = wave + u * kTnWaves;
            if (S::CHUNKS % kTnWaves && chunk >= S::CHUNKS) break;
            const unsigned flip = chunk % (S::COLS / kWave) < S::MT / kWave ? sign : 0u;
            bf16_words4 w[3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                unsigned p[3];
                bf16_split2(f[u][2 * i], f[u][2 * i + 1], p);
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
    unsigned sign = blockIdx.x & 1 ? 0x80008000u : 0u;    // of the stage being multiplied
    fetch(0);
    park(0, sign);
    __syncthreads();
    int buf = 0;
    for (int r0 = 0; r0 < rows; r0 += 16 * S::KB) {
        const bool more = r0 + 16 * S::KB < rows;
        if (more) fetch(r0 + 16 * S::KB);
        const float factor = sign ? -1.f : 1.f;
#pragma unroll
        for (int kb = 0; kb < S::KB / S::KW; ++kb) {
            const bf16_words4* src = words + buf * 3 * S::PIECE + (2 * (kb * S::KW + kw) + (lane >> 5)) * S::COLS + (lane & 31);
            auto load_a = [&](int i, bf16_words4 (&a)[3]) {
#pragma unroll
                for (int p = 0; p < 3; ++p) a[p] = src[p * S::PIECE + (wr * S::TR + i) * 32];
            };
            bf16_words4 a[S::KEEP_A ? S::TR : 1][3];
            if (S::KEEP_A) {
#pragma unroll
                for (int i = 0; i < S::TR; ++i) load_a(i, a[i]);
            }
#pragma unroll
            for (int j = 0; j < S::TC; ++j) {
                bf16_words4 b[3];
#pragma unroll
                for (int p = 0; p < 3; ++p) b[p] = src[p * S::PIECE + S::MT + (wc * S::TC + j) * 32];
#pragma unroll
                for (int i0 = 0; i0 < S::TR; i0 += S::SUMS) {
                    mfma_f16 sum[S::SUMS];
#pragma unroll
                    for (int i = 0; i < S::SUMS; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) sum[i][r] = 0.f;
                    if (!S::KEEP_A) load_a(i0, a[0]);
#pragma unroll
                    for (int p = 2; p >= 0; --p)
#pragma unroll
                        for (int o = 2 - p; o >= 0; --o)
#pragma unroll
                            for (int i = 0; i < S::SUMS; ++i) {
                                const bf16_words4& x = a[S::KEEP_A ? i0 + i : 0][o];
                                sum[i] = TRANSPOSED ? mfma_32(b[p], x, sum[i]) : mfma_32(x, b[p], sum[i]);
                            }
#pragma unroll
                    for (int i = 0; i < S::SUMS; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[i0 + i][j][r] = fmaf(sum[i][r], factor, acc[i0 + i][j][r]);
                    // the sums are added here: the compiler would gather the additions of all tiles behind the last product, and
                    // that many sums do not fit the registers
#pragma unroll
                    for (int i = 0; i < S::SUMS; ++i) asm volatile("" : "+v"(acc[i0 + i][j]));
                }
            }
        }
        sign ^= 0x80008000u;
        if (more) park(buf ^ 1, sign);
        __syncthreads();
        buf ^= 1;
    }

    // lane l ends with column l % 32 of a tile (of its transpose) and rows 8 (r / 4) + 4 (l / 32) + r % 4
    float* part = partial + ((size_t)blockIdx.x * S::KW + kw) * m * n;
#pragma unroll
    for (int i = 0; i < S::TR; ++i)
#pragma unroll
        for (int j = 0; j < S::TC; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int x = lane & 31, y = 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
                const int row = (wr * S::TR + i) * 32 + (TRANSPOSED ? x : y), col = (wc * S::TC + j) * 32 + (TRANSPOSED ? y : x);
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
    if (m <= 128) GNNHIP_TN(128, 256, 2, 4, 1, 1);
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
