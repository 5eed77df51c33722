// Dense fp32 GEMM for gfx950:  C[m,n] = alpha * op(A) * op(B) + beta * C, row-major.
//
// The mean-field path only has tall-and-skinny products (m = nodes or graphs,
// n and k = label types / hidden sizes <= 256), which are HBM-bound: every A
// element is used n times from LDS, every B element lives in L2.  The kernel is
// an LDS-tiled SGEMM on the FP32 matrix cores: a 64 x 64 output tile per 256-lane
// workgroup, 16 rows x 64 columns per wavefront as four v_mfma_f32_16x16x4_f32
// accumulators, K walked in steps of 16 through two LDS tiles.  Edges are handled
// by bounds-checked tile loads (zeros) and stores.
// Bound: HBM for the shapes above; algorithmic bytes 4(mk + kn + mn).
//
// Weight gradients are the opposite shape: op(A)^T * G with a small output (hidden x hidden) and k = nodes.
// One output tile would walk all of k on one CU (1.1 ms at k = 7,450; 15 us at k = 256, a microsecond per step of 16),
// so such products are split along k from k = 256:
// every workgroup takes a range of k, writes its partial tile to scratch, and a second kernel adds the
// partial tiles in range order (deterministic) and applies alpha and beta.
#include <algorithm>
#include <limits.h>

#include "columns.h"

namespace gnnhip {
namespace {

constexpr int BM = 64, BN = 64, BK = 16, kBlock = 256;

// One 64 x 64 output tile (tile_x, tile_y) over k in [k_lo, k_hi).  part != nullptr: the raw sums go to
// part[m][n]; otherwise the tile finishes C itself.
template <bool TA, bool TB>
__device__ __forceinline__ void sgemm_tile_body(
    int m, int n, float alpha, const float* __restrict__ A, int lda,
    const float* __restrict__ B, int ldb, float beta, float* C, int ldc, int k_lo, int k_hi, float* __restrict__ part,
    int tile_x, int tile_y)
{
    // Both tiles sit in LDS with k contiguous, so that a lane fetches its four k values of a step with one
    // 128-bit read.  Wavefront w owns the output rows 16 w .. 16 w + 15 of the tile and all 64 columns: four
    // accumulators of v_mfma_f32_16x16x4_f32 with the operand roles swapped (out^T = B^T * A^T), which leaves
    // lane (q = lane/16, t = lane%16) with row t and the columns 16 jb + 4 q .. + 3 of block jb.
    constexpr int LD = BK + 4;
    __shared__ float As[BM][LD];         // As[i][p] = op(A)[row0 + i][k0 + p]
    __shared__ float Bs[BN][LD];         // Bs[j][p] = op(B)[k0 + p][col0 + j]

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    const int q = lane >> 4, t = lane & 15;
    const long long row0 = (long long)tile_x * BM;
    const int col0 = tile_y * BN;

    mfma_f4 acc[BN / 16];
#pragma unroll
    for (int jb = 0; jb < BN / 16; ++jb) acc[jb] = mfma_f4{0.f, 0.f, 0.f, 0.f};

    // each lane moves 4 elements of each tile; the elements of the next step are requested before the products of this one are
    // formed, so a step costs the longer of the two instead of their sum
    float ra[4], rb[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int idx = tid + e * kBlock;        // 0 .. 1023
            {
                // A tile: the fast index follows memory
                int i, p;
                if (TA) { i = idx & (BM - 1); p = idx >> 6; }       // stored A is [k][m]: i contiguous
                else    { p = idx & (BK - 1); i = idx >> 4; }       // stored A is [m][k]: p contiguous
                const long long gi = row0 + i;
                const int gp = k0 + p;
                float v = 0.f;
                if (gi < m && gp < k_hi) v = TA ? A[(size_t)gp * lda + gi] : A[(size_t)gi * lda + gp];
                ra[e] = v;
            }
            {
                int j, p;
                if (TB) { p = idx & (BK - 1); j = idx >> 4; }       // stored B is [n][k]: p contiguous
                else    { j = idx & (BN - 1); p = idx >> 6; }       // stored B is [k][n]: j contiguous
                const int gj = col0 + j;
                const int gp = k0 + p;
                float v = 0.f;
                if (gj < n && gp < k_hi) v = TB ? B[(size_t)gj * ldb + gp] : B[(size_t)gp * ldb + gj];
                rb[e] = v;
            }
        }
    };
    fetch(k_lo);
    for (int k0 = k_lo; k0 < k_hi; k0 += BK) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int idx = tid + e * kBlock;
            if (TA) As[idx & (BM - 1)][idx >> 6] = ra[e]; else As[idx >> 4][idx & (BK - 1)] = ra[e];
            if (TB) Bs[idx >> 4][idx & (BK - 1)] = rb[e]; else Bs[idx & (BN - 1)][idx >> 6] = rb[e];
        }
        __syncthreads();
        if (k0 + BK < k_hi) fetch(k0 + BK);
        // lane (q, t): k = 4 q + s at instruction s of the step
        const float4 a = *reinterpret_cast<const float4*>(&As[wave * 16 + t][4 * q]);
#pragma unroll
        for (int jb = 0; jb < BN / 16; ++jb) {
            const float4 b = *reinterpret_cast<const float4*>(&Bs[jb * 16 + t][4 * q]);
            acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.x, a.x, acc[jb], 0, 0, 0);
            acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.y, a.y, acc[jb], 0, 0, 0);
            acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.z, a.z, acc[jb], 0, 0, 0);
            acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.w, a.w, acc[jb], 0, 0, 0);
        }
        __syncthreads();
    }

    // lane (q, t) holds out[row0 + 16 wave + t][col0 + 16 jb + 4 q + i], i = 0..3
    const long long gi = row0 + wave * 16 + t;
    if (gi < m) {
#pragma unroll
        for (int jb = 0; jb < BN / 16; ++jb) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int gj = col0 + jb * 16 + 4 * q + i;
                if (gj >= n) continue;
                if (part) {
                    part[(size_t)gi * n + gj] = acc[jb][i];
                    continue;
                }
                float* dst = C + (size_t)gi * ldc + gj;
                const float r = alpha * acc[jb][i];
                *dst = (beta == 0.f) ? r : r + beta * (*dst);
            }
        }
    }
}

// partial != nullptr: workgroup z handles k in [z k_chunk, (z+1) k_chunk) and stores its raw sums to
// partial[z][m][n]; otherwise one workgroup walks all of k and finishes C itself.
template <bool TA, bool TB>
__global__ __launch_bounds__(kBlock) void sgemm_tile_kernel(
    int m, int n, int k, float alpha, const float* __restrict__ A, int lda,
    const float* __restrict__ B, int ldb, float beta, float* C, int ldc, int k_chunk, float* __restrict__ partial)
{
    const int k_lo = partial ? (int)blockIdx.z * k_chunk : 0;
    const int k_hi = partial ? min(k, k_lo + k_chunk) : k;
    sgemm_tile_body<TA, TB>(m, n, alpha, A, lda, B, ldb, beta, C, ldc, k_lo, k_hi,
                            partial ? partial + (size_t)blockIdx.z * m * n : nullptr, (int)blockIdx.x, (int)blockIdx.y);
}

// ---- A^T B: op(A) = A^T with A stored [k][m], B stored [k][n] (weight gradients, alone or several at the end of a backward pass)
//
// Four rows of k of either operand are what v_mfma_f32_16x16x4_f32 takes, and both lie in memory as it wants them: lane
// (q = lane/16, t = lane%16) loads columns 4 t .. 4 t + 3 of row q in one 128-bit word, and word j of all lanes is the
// operand of the block of columns {4 t + j}.  So a step of four rows is two loads and sixteen matrix instructions for a
// 64 x 64 tile, without LDS and without a barrier; the four wavefronts of a workgroup take four rows of sixteen each and add
// up their tiles in wavefront order at the end.  An output tile ends with a lane holding four consecutive columns.
// What bounds it at the sizes of a training batch is one or two trips to memory, the sum over the wavefronts and the launch: with the
// sums of the ranges 7,450 nodes x 4 levels at hidden 64 (four products) take 13.5 us, 1,625 x 3 8.4 (LDS tiles and a
// barrier per sixteen rows: 20.4 and 11.4); 1,000 x 500 over 3,000 rows 57 (128), 2,048^3 178 = 96 TFLOP/s (210).
// Six steps under way: four take 0.3 to 1 us more where a range is short, eight spill.
constexpr int kTnWaves = kBlock / kWave;
constexpr int kTnStep = 4 * kTnWaves;        // rows of k per step of the workgroup
constexpr int kTnAhead = 6;                  // steps under way

// Output tile (tile_x, tile_y), rows [k_lo, k_hi).  part != nullptr: the sums go to part[m][n]; otherwise the tile finishes C.
// A tile narrower than 64 moves its last unit of four columns back to end with it (the columns that repeat have the same
// sums twice, and one owner where C is updated); NA, NB: fewer than four columns of A, of B, read one by one.
template <bool NA, bool NB>
__device__ __forceinline__ void tn_tile_body(int m, int n, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ B,
                                             int ldb, float beta, float* C, int ldc, int k_lo, int k_hi, float* __restrict__ part,
                                             int tile_x, int tile_y, float4 (&sums)[kTnWaves - 1][4][4][kWave])
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int wa = min(m - tile_x * BM, BM), wb = min(n - tile_y * BN, BN);          // columns of the operands in this tile
    auto unit_a = [&](int u) { return NA ? 0 : min(4 * u, wa - 4); };
    auto unit_b = [&](int u) { return NB ? 0 : min(4 * u, wb - 4); };
    const float* a_col = A + (size_t)tile_x * BM + unit_a(t);
    const float* b_col = B + (size_t)tile_y * BN + unit_b(t);
    auto few = [](const float* p, int w) { return make_float4(p[0], w > 1 ? p[1] : 0.f, w > 2 ? p[2] : 0.f, 0.f); };
    auto row_a = [&](size_t k) { const float* p = a_col + k * lda; if constexpr (NA) return few(p, wa); else return ColsLoose::load(p); };
    auto row_b = [&](size_t k) { const float* p = b_col + k * ldb; if constexpr (NB) return few(p, wb); else return ColsLoose::load(p); };

    mfma_f4 acc[4][4];                          // [block of A][block of B]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma_f4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](const float4& a4, const float4& b4) {
        const float a[4] = {a4.x, a4.y, a4.z, a4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
    };

    const int steps = (k_hi - k_lo) / kTnStep;
    const size_t k0 = (size_t)k_lo + 4 * wave + q;
    float4 a[kTnAhead], b[kTnAhead];
#pragma unroll
    for (int d = 0; d < kTnAhead; ++d)
        if (d < steps) { a[d] = row_a(k0 + d * kTnStep); b[d] = row_b(k0 + d * kTnStep); }
    // the rows short of a step: a row past the end is read as zeros (of both operands: 0 times an infinity is none)
    const int rest = k_lo + steps * kTnStep + 4 * wave;         // this wavefront's first of them
    float4 al = f4_zero(), bl = f4_zero();
    if (rest + q < k_hi) { al = row_a((size_t)rest + q); bl = row_b((size_t)rest + q); }
    int s = 0;
    for (; s + kTnAhead <= steps; s += kTnAhead) {
#pragma unroll
        for (int d = 0; d < kTnAhead; ++d) {
            products(a[d], b[d]);
            const int ahead = s + d + kTnAhead;
            if (ahead < steps) { a[d] = row_a(k0 + (size_t)ahead * kTnStep); b[d] = row_b(k0 + (size_t)ahead * kTnStep); }
        }
    }
#pragma unroll
    for (int d = 0; d < kTnAhead - 1; ++d)
        if (s + d < steps) products(a[d], b[d]);
    if (rest < k_hi) products(al, bl);

    // wavefront w adds up block w of A over the four wavefronts
    mfma_f4 own[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i == wave) {
#pragma unroll
            for (int j = 0; j < 4; ++j) own[j] = acc[i][j];
        } else {
            const int slot = wave < i ? wave : wave - 1;
#pragma unroll
            for (int j = 0; j < 4; ++j) sums[slot][i][j][lane] = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        }
    }
    __syncthreads();
    float out[4][4];                            // [row][column] of this lane
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float4 v[kTnWaves - 1];
#pragma unroll
        for (int w = 0; w < kTnWaves - 1; ++w) v[w] = sums[w][wave][j][lane];
        mfma_f4 total = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kTnWaves; ++w) {
            if (w == wave) total += own[j];
            else {
                const float4 x = v[w < wave ? (w < kTnWaves - 1 ? w : 0) : (w > 0 ? w - 1 : 0)];
                total += mfma_f4{x.x, x.y, x.z, x.w};
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i][j] = total[i];
    }
    // out[i][j]: row unit_a(4 q + i) + wave, column unit_b(t) + j of the tile
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int u = 4 * q + i, r = unit_a(u) + wave;
        if (NA ? u > 0 || wave >= wa : r < 4 * u) continue;                  // a unit past the tile, or a row that an earlier unit has
        const size_t gi = (size_t)tile_x * BM + r;
        const int c = unit_b(t), gj = tile_y * BN + c;
        if (NB ? t > 0 : 4 * t >= wb) continue;
        if (!NB && part) {
            ColsLoose::store(part + gi * n + gj, make_float4(out[i][0], out[i][1], out[i][2], out[i][3]));
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (NB ? j >= wb : c + j < 4 * t) continue;
            if (part) { part[gi * n + gj + j] = out[i][j]; continue; }
            float* dst = C + gi * ldc + gj + j;
            const float v = alpha * out[i][j];
            *dst = (beta == 0.f) ? v : v + beta * (*dst);
        }
    }
}

// The same for few rows of k: nothing to share out between the wavefronts, whose tiles would only have to be added up
// again.  Each takes sixteen columns of A instead, asks for all its rows (ROWS at most) at once and finishes its rows of C; no LDS, no
// barrier, and nothing is read for columns that are not there.  A product alone is launched without the 48 KB of LDS that the sums above
// take: 16 rows, 16 x 16 3.8 -> 2.2 us, 38 x 64 3.8 -> 3.3, 1,000 x 500 4.5 -> 3.9.  The line lies at 32 rows, and at 48 for outputs of
// up to 1,024 elements (48 rows, 16 x 16: 4.6 -> 3.2; 38 x 64: 4.2 -> 4.7).
constexpr int kTnShort = 32, kTnShortSmall = 48;
inline bool tn_short(int m, int n, int k) { return k <= ((long long)m * n <= 1024 ? kTnShortSmall : kTnShort); }
template <int ROWS>
__device__ __forceinline__ void tn_short_body(int m, int n, int k, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ B,
                                              int ldb, float beta, float* C, int ldc, int tile_x, int tile_y)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int q = lane >> 4, t = lane & 15;
    const int row0 = tile_x * BM + 16 * wave, col0 = tile_y * BN;
    if (row0 >= m) return;
    const float* a_col = A + min(row0 + t, m - 1);
    float a[ROWS / 4], b[ROWS / 4][BN / 16];
#pragma unroll
    for (int g = 0; g < ROWS / 4; ++g) {
        if (4 * g >= k) break;                                  // uniform, as is every test of a block of columns
        const int r = 4 * g + q;                                // a row past k is read as zeros (of both operands)
        a[g] = r < k ? a_col[(size_t)r * lda] : 0.f;
#pragma unroll
        for (int j = 0; j < BN / 16; ++j)
            if (col0 + 16 * j < n) b[g][j] = r < k ? B[(size_t)r * ldb + min(col0 + 16 * j + t, n - 1)] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < BN / 16; ++j) {
        if (col0 + 16 * j >= n) break;
        mfma_f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < ROWS / 4; ++g)
            if (4 * g < k) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[g], b[g][j], acc, 0, 0, 0);
        const int gj = col0 + 16 * j + t;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int gi = row0 + 4 * q + i;
            if (gi >= m || gj >= n) continue;
            float* dst = C + (size_t)gi * ldc + gj;
            const float v = alpha * acc[i];
            *dst = (beta == 0.f) ? v : v + beta * (*dst);
        }
    }
}

// Several products C_p = alpha A_p^T B_p + beta C_p in one launch.  Product p owns the z range [z0[p], z0[p+1]) of the
// grid, one range of k per z; tiles outside a product's own tile grid leave at once.
constexpr int kGemmBatch = 8;
struct GemmJob {                                // a cache line of the kernel's arguments each
    const float* A;
    const float* B;
    float* C;
    float* partial;                             // null: one range, finished by the product launch
    int m, n, k, lda, ldb, ldc;
    int k_chunk;                                // 0: tn_short
    int splits;
};
struct GemmBatch {
    int z0[kGemmBatch];                         // INT_MAX from `count` on
    GemmJob job[kGemmBatch];
    int count;
};

template <int ROWS>
__global__ __launch_bounds__(kBlock) void sgemm_tn_short_kernel(GemmJob j, float alpha, float beta)
{
    tn_short_body<ROWS>(j.m, j.n, j.k, alpha, j.A, j.lda, j.B, j.ldb, beta, j.C, j.ldc, (int)blockIdx.x, (int)blockIdx.y);
}

// SHORT: some of the products may be short ones
template <bool SHORT>
__global__ __launch_bounds__(kBlock, 3) void sgemm_tn_batch_kernel(GemmBatch b, float alpha, float beta)
{
    __shared__ float4 sums[kTnWaves - 1][4][4][kWave];        // [wavefront other than a block's owner][block of A][block of B][lane]
    int p = 0;
#pragma unroll
    for (int i = 1; i < kGemmBatch; ++i) p += (int)blockIdx.z >= b.z0[i];
    const GemmJob j = b.job[p];
    const int m = j.m, n = j.n;
    if ((long long)blockIdx.x * BM >= m || (int)blockIdx.y * BN >= n) return;
    if (SHORT && j.k_chunk == 0) {
        tn_short_body<kTnShortSmall>(m, n, j.k, alpha, j.A, j.lda, j.B, j.ldb, beta, j.C, j.ldc, (int)blockIdx.x, (int)blockIdx.y);
        return;
    }
    const int z = (int)blockIdx.z - b.z0[p];
    const int k_lo = z * j.k_chunk, k_hi = min(j.k, k_lo + j.k_chunk);
    float* part = j.partial ? j.partial + (size_t)z * m * n : nullptr;
    const bool na = m - (int)blockIdx.x * BM < 4, nb = n - (int)blockIdx.y * BN < 4;
#define GNNHIP_TN_BODY(NA, NB) \
    tn_tile_body<NA, NB>(m, n, alpha, j.A, j.lda, j.B, j.ldb, beta, j.C, j.ldc, k_lo, k_hi, part, (int)blockIdx.x, (int)blockIdx.y, sums)
    if (!na && !nb) GNNHIP_TN_BODY(false, false);
    else if (!na) GNNHIP_TN_BODY(false, true);
    else if (!nb) GNNHIP_TN_BODY(true, false);
    else GNNHIP_TN_BODY(true, true);
#undef GNNHIP_TN_BODY
}

// C = alpha * (sum over z of partial[z]) + beta * C.  A workgroup takes 64 consecutive elements, four to a lane: group g of
// sixteen lanes adds the ranges z = g, g + 16, ... (up to eight 128-bit loads in flight per lane) and the sixteen sums are added in group order, so
// the result is the same on every run.  The additions are in double: with up to 1,024 ranges an fp32
// sum of theirs had a larger error than the ranges themselves (64 x 64 over 70,000 rows, terms of one sign: rms 9.5e-8 of the
// sum, 2.5e-8 in double).  The kernel reads memory meanwhile; it takes the same time.
__device__ __forceinline__ void sgemm_splitk_reduce_body(int m, int n, int splits, float alpha,
                                                         const float* __restrict__ partial, float beta,
                                                         float* C, int ldc)
{
    constexpr int kGroups = kBlock / 16, kBatch = 8;
    __shared__ double part[kGroups][kWave];
    const size_t total = (size_t)m * n;
    const int tid = threadIdx.x, group = tid >> 4, e = tid & 15;
    for (size_t base = (size_t)blockIdx.x * kWave; base < total; base += (size_t)gridDim.x * kWave) {
        const int width = (int)min(total - base, (size_t)kWave);
        const size_t idx = base + tid;
        float* dst = nullptr;
        float c_old = 0.f;
        if (tid < width) {
            dst = C + (idx / n) * (size_t)ldc + idx % n;
            if (beta != 0.f) c_old = *dst;                      // asked for before the sums, not after
        }
        if (width >= 4) {
            // (the last unit is moved back to end with the elements: those that repeat have the same sums twice)
            const int at = min(4 * e, width - 4);
            const float* src = partial + (size_t)group * total + base + at;
            double s[4] = {0.0, 0.0, 0.0, 0.0};
            auto add = [&](const float4& x) { s[0] += x.x; s[1] += x.y; s[2] += x.z; s[3] += x.w; };
            const size_t step = (size_t)kGroups * total;
            int z = group;
            for (; z + (kBatch - 1) * kGroups < splits; z += kBatch * kGroups, src += kBatch * step) {
                float4 x[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) x[u] = ColsLoose::load(src + u * step);
#pragma unroll
                for (int u = 0; u < kBatch; ++u) add(x[u]);
            }
            for (; z + kGroups < splits; z += 2 * kGroups, src += 2 * step) {
                const float4 x0 = ColsLoose::load(src), x1 = ColsLoose::load(src + step);
                add(x0);
                add(x1);
            }
            if (z < splits) add(ColsLoose::load(src));
#pragma unroll
            for (int i = 0; i < 4; ++i) part[group][at + i] = s[i];
        } else if (e < width) {
            double s = 0.0;
            for (int z = group; z < splits; z += kGroups) s += partial[(size_t)z * total + base + e];
            part[group][e] = s;
        }
        __syncthreads();
        if (tid < width) {
            double t = part[0][tid];
#pragma unroll
            for (int g = 1; g < kGroups; ++g) t += part[g][tid];
            const float r = alpha * (float)t;
            *dst = (beta == 0.f) ? r : r + beta * c_old;
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void sgemm_splitk_reduce_kernel(int m, int n, int splits, float alpha,
                                                                     const float* __restrict__ partial, float beta,
                                                                     float* C, int ldc)
{
    sgemm_splitk_reduce_body(m, n, splits, alpha, partial, beta, C, ldc);
}

// the sums of product blockIdx.y of a batch
__global__ __launch_bounds__(kBlock) void sgemm_splitk_reduce_batch_kernel(GemmBatch b, float alpha, float beta)
{
    const GemmJob j = b.job[blockIdx.y];
    if (j.partial) sgemm_splitk_reduce_body(j.m, j.n, j.splits, alpha, j.partial, beta, j.C, j.ldc);
}

}  // namespace

namespace {

// ---- tall A times a matrix of at most four columns (node scores h * w, readouts with one or two
// classes): a group of G lanes walks one row of A in 128-bit pieces and reduces with shuffles.
// Reads A once at streaming rate; the tile kernel would spend a 64-column tile on it.
template <int NCOL, bool TB>
__global__ __launch_bounds__(kBlock) void sgemm_skinny_kernel(
    int m, int k, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
    float beta, float* C, int ldc, int logG)
{
    const int G = 1 << logG;
    const int sub = threadIdx.x & (G - 1);
    const long long row = ((long long)blockIdx.x * kBlock + threadIdx.x) >> logG;
    float acc[NCOL];
#pragma unroll
    for (int j = 0; j < NCOL; ++j) acc[j] = 0.f;
    if (row < m) {
        const float* a = A + (size_t)row * lda;
        for (int kk = sub * 4; kk < k; kk += G * 4) {
            const float4 x = *reinterpret_cast<const float4*>(a + kk);
#pragma unroll
            for (int j = 0; j < NCOL; ++j) {
                const float b0 = TB ? B[(size_t)j * ldb + kk] : B[(size_t)kk * ldb + j];
                const float b1 = TB ? B[(size_t)j * ldb + kk + 1] : B[(size_t)(kk + 1) * ldb + j];
                const float b2 = TB ? B[(size_t)j * ldb + kk + 2] : B[(size_t)(kk + 2) * ldb + j];
                const float b3 = TB ? B[(size_t)j * ldb + kk + 3] : B[(size_t)(kk + 3) * ldb + j];
                acc[j] += x.x * b0 + x.y * b1 + x.z * b2 + x.w * b3;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NCOL; ++j)
        for (int d = G >> 1; d >= 1; d >>= 1) acc[j] += __shfl_xor(acc[j], d, kWave);
    if (row < m && sub == 0) {
#pragma unroll
        for (int j = 0; j < NCOL; ++j) {
            float* c = C + (size_t)row * ldc + j;
            *c = (beta == 0.f) ? alpha * acc[j] : alpha * acc[j] + beta * *c;
        }
    }
}

// The same product for k <= 256: a lane keeps its four rows of B in registers, the groups stride the rows of A
// eight at a time (eight 128-bit loads in flight per lane), and groups of up to 16 lanes reduce with DPP.
// LOOSE: rows of any alignment and length; the row's last lane reads its last four columns (columns.h) and counts only its own
// (1M rows of 53: 99 us with the tile kernel, 33 here).
template <int NCOL, bool TB, bool LOOSE>
__global__ __launch_bounds__(kBlock) void sgemm_skinny_rows_kernel(
    int m, int k, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
    float beta, float* C, int ldc, int logG)
{
    constexpr int R = 8;
    const int G = 1 << logG;
    const int sub = threadIdx.x & (G - 1);
    const bool live = sub * 4 < k;
    const int kk = LOOSE ? ColsLoose::at(sub, k) : sub * 4;
    const int skip = sub * 4 - kk;                         // columns of the lane before
    float4 b[NCOL];
#pragma unroll
    for (int j = 0; j < NCOL; ++j) {
        b[j] = f4_zero();
        if (live) {
            b[j].x = TB ? B[(size_t)j * ldb + kk] : B[(size_t)kk * ldb + j];
            b[j].y = TB ? B[(size_t)j * ldb + kk + 1] : B[(size_t)(kk + 1) * ldb + j];
            b[j].z = TB ? B[(size_t)j * ldb + kk + 2] : B[(size_t)(kk + 2) * ldb + j];
            b[j].w = TB ? B[(size_t)j * ldb + kk + 3] : B[(size_t)(kk + 3) * ldb + j];
        }
        if (LOOSE) {                                       // both factors of a repeated column are zeros: either may be infinite
            if (skip > 0) b[j].x = 0.f;
            if (skip > 1) b[j].y = 0.f;
            if (skip > 2) b[j].z = 0.f;
        }
    }
    // A workgroup walks one contiguous run of rows (its groups side by side, R turns ahead), so that what is in flight
    // from one workgroup is one stretch of memory.  All lanes of a wavefront run the same number of iterations (the
    // reductions are wavefront-wide operations).
    const int groups = kBlock >> logG;
    const int group = threadIdx.x >> logG;
    const long long per_block = ((long long)m + gridDim.x - 1) / gridDim.x;
    const long long row0 = (long long)blockIdx.x * per_block;
    const long long row1 = row0 + per_block < m ? row0 + per_block : m;
    for (long long base = row0; base < row1; base += R * groups) {
        float4 x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const long long row = base + r * groups + group;
            if (!LOOSE) {
                x[r] = (live && row < row1) ? ColsWide::load(A + (size_t)row * lda + kk) : f4_zero();
            } else {
                x[r] = (live && row < row1) ? ColsLoose::load(A + (size_t)row * lda + kk) : f4_zero();
                if (skip > 0) x[r].x = 0.f;
                if (skip > 1) x[r].y = 0.f;
                if (skip > 2) x[r].z = 0.f;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const long long row = base + r * groups + group;
#pragma unroll
            for (int j = 0; j < NCOL; ++j) {
                float acc = x[r].x * b[j].x + x[r].y * b[j].y + x[r].z * b[j].z + x[r].w * b[j].w;
                if (G >= 2) acc += dpp_mov_f<kDppXor1>(acc);
                if (G >= 4) acc += dpp_mov_f<kDppXor2>(acc);
                if (G >= 8) acc += dpp_mov_f<kDppHalfMirror>(acc);
                if (G >= 16) acc += dpp_mov_f<kDppMirror>(acc);
                if (G >= 32) acc += __shfl_xor(acc, 16, kWave);
                if (G >= 64) acc += __shfl_xor(acc, 32, kWave);
                if (row < row1 && sub == 0) {
                    float* c = C + (size_t)row * ldc + j;
                    *c = (beta == 0.f) ? alpha * acc : alpha * acc + beta * *c;
                }
            }
        }
    }
}

template <int NCOL>
void launch_skinny(bool tb, bool loose, int m, int k, float alpha, const float* A, int lda, const float* B, int ldb,
                   float beta, float* C, int ldc, hipStream_t s)
{
    int logG = 0;
    while ((4 << logG) < k && logG < 6) ++logG;              // G * 4 >= k, at most one wavefront per row
    if (k <= 4 * kWave) {
        const size_t lanes = (size_t)m << logG;
        size_t blocks = ceil_div_u(ceil_div_u(lanes, 8), kBlock);          // eight rows per group
        if (blocks > (size_t)kNumCU * 32) blocks = (size_t)kNumCU * 32;
        if (blocks < 1) blocks = 1;
        const unsigned grid = (unsigned)blocks;
        const auto kernel = loose ? (tb ? sgemm_skinny_rows_kernel<NCOL, true, true> : sgemm_skinny_rows_kernel<NCOL, false, true>)
                                  : (tb ? sgemm_skinny_rows_kernel<NCOL, true, false> : sgemm_skinny_rows_kernel<NCOL, false, false>);
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, s, m, k, alpha, A, lda, B, ldb, beta, C, ldc, logG);
        return;
    }
    const unsigned grid = ceil_div_u((size_t)m << logG, kBlock);
    if (tb) hipLaunchKernelGGL((sgemm_skinny_kernel<NCOL, true>), dim3(grid), dim3(kBlock), 0, s, m, k, alpha, A, lda, B, ldb, beta, C, ldc, logG);
    else hipLaunchKernelGGL((sgemm_skinny_kernel<NCOL, false>), dim3(grid), dim3(kBlock), 0, s, m, k, alpha, A, lda, B, ldb, beta, C, ldc, logG);
}

}  // namespace

// gemm_tn_split.hip: outputs of up to 256 x 256 over a very long k
int gemm_tn_split_dispatch(int m, int n, int k, float alpha, const float* A, int lda, const float* B, int ldb, float beta, float* C,
                          int ldc, hipStream_t s);

void launch_splitk_reduce(int m, int n, int splits, float alpha, const float* partial, float beta, float* C, int ldc, hipStream_t s)
{
    const size_t total = (size_t)m * n;
    const unsigned rgrid = ceil_div_u(total, kWave) < 2048u ? ceil_div_u(total, kWave) : 2048u;
    hipLaunchKernelGGL(sgemm_splitk_reduce_kernel, dim3(rgrid), dim3(kBlock), 0, s, m, n, splits, alpha, partial, beta, C, ldc);
}

// length of the ranges of k when few output tiles share a long k: about two workgroups per CU, four steps at least
inline long long splitk_chunk(long long tiles, long long k)
{
    const long long want = (2 * kNumCU) / tiles;                           // ranges per tile
    long long chunk = (k + want - 1) / want;
    if (chunk < 4 * BK) chunk = 4 * BK;
    return (chunk + BK - 1) / BK * BK;
}
// The same for A^T B: a workgroup per CU, two steps of its four wavefronts at least.  (64 x 64 over 60,000 rows: 14.8 us with one,
// 17.8 with two per CU, whose partial tiles are twice as many, 18.4 with one per two CUs; ranges of at least 128 rows cost
// batches of up to 7,450 nodes 0.6 to 1.5 us.)
inline long long tn_chunk(long long tiles, long long k)
{
    const long long want = kNumCU / tiles;                                 // tiles <= kNumCU / 4
    const long long chunk = std::max((k + want - 1) / want, 2ll * kTnStep);
    return (chunk + kTnStep - 1) / kTnStep * kTnStep;
}

// count <= kGemmBatch products C_p = alpha A_p^T B_p + beta C_p (A_p stored [k_p, m_p], B_p [k_p, n_p]) in two launches
int gemm_tn_batch_dispatch(int count, const int* m, const int* n, const int* k, const float* const* A, const int* lda,
                           const float* const* B, const int* ldb, float alpha, float beta, float* const* C, const int* ldc, hipStream_t s)
{
    GemmBatch b;
    b.count = 0;
    size_t floats = 0;
    unsigned gx = 1, gy = 1, red = 0;
    constexpr size_t kDirect = ~(size_t)0;
    size_t offset[kGemmBatch];
    int z = 0;
    for (int p = 0; p < count; ++p) {
        if (m[p] == 0 || n[p] == 0) continue;
        // the rule of the single product here too: an output of up to 256 x 256 over a very long k has a kernel of its own
        if (int rc = gemm_tn_split_dispatch(m[p], n[p], k[p], alpha, A[p], lda[p], B[p], ldb[p], beta, C[p], ldc[p], s);
            rc != GNNHIP_EUNSUPPORTED) {
            if (rc) return rc;
            continue;
        }
        const int q = b.count++;
        const unsigned tx = ceil_div_u((size_t)m[p], BM), ty = ceil_div_u((size_t)n[p], BN);
        const long long tiles = (long long)tx * ty;
        // the rule of the single product, so that a batch gives the bits of its products done one by one
        long long chunk = tiles <= kNumCU / 4 && k[p] >= 256 ? tn_chunk(tiles, k[p]) : (k[p] > 0 ? k[p] : 1);
        const int splits = k[p] > 0 ? (int)(((long long)k[p] + chunk - 1) / chunk) : 1;
        b.job[q] = GemmJob{A[p], B[p], C[p], nullptr, m[p], n[p], k[p], lda[p], ldb[p], ldc[p], tn_short(m[p], n[p], k[p]) ? 0 : (int)chunk, splits};
        b.z0[q] = z;
        z += splits;
        offset[q] = splits > 1 ? floats : kDirect;
        if (splits > 1) floats += (size_t)splits * m[p] * n[p];
        if (tx > gx) gx = tx;
        if (ty > gy) gy = ty;
        if (splits > 1) red = std::max(red, std::min(ceil_div_u((size_t)m[p] * n[p], kWave), 2048u));
    }
    if (b.count == 0) return GNNHIP_OK;
    if (b.count == 1 && b.job[0].k_chunk == 0) {
        hipLaunchKernelGGL(b.job[0].k <= kTnShort ? sgemm_tn_short_kernel<kTnShort> : sgemm_tn_short_kernel<kTnShortSmall>, dim3(gx, gy), dim3(kBlock), 0, s,
                           b.job[0], alpha, beta);
        GNNHIP_LAUNCH_CHECK("sgemm_tn_short");
        return GNNHIP_OK;
    }
    for (int p = b.count; p < kGemmBatch; ++p) b.z0[p] = INT_MAX;
    void* q = nullptr;
    if (floats)
        if (int rc = stream_scratch_slot(s, 2, sizeof(float) * floats, &q)) return rc;
    for (int p = 0; p < b.count; ++p) b.job[p].partial = offset[p] == kDirect ? nullptr : static_cast<float*>(q) + offset[p];
    // The two variants differ in what the compiler makes of the long products, too: the one without the short body starts sooner (64 x 64 over
    // 200 rows 7.1 us, 7.3 with it; 7,450 nodes x 4 levels 13.5, 13.7), the other one is ahead where tiles follow each other on a
    // compute unit (2,000^2 over 200 rows 35.0, 30.0; over 1,000 94.3, 92.9), from some two per compute unit on; 1,200^2 is even.
    // Over 48 to 64 rows that one is 2 to 3 % behind at any size.
    bool with_short = false;
    for (int p = 0; p < b.count; ++p) with_short |= b.job[p].k_chunk == 0 || (b.job[p].k >= 128 && (long long)gx * gy > 2 * kNumCU);
    hipLaunchKernelGGL(with_short ? sgemm_tn_batch_kernel<true> : sgemm_tn_batch_kernel<false>, dim3(gx, gy, (unsigned)z), dim3(kBlock), 0, s, b, alpha, beta);
    if (red) hipLaunchKernelGGL(sgemm_splitk_reduce_batch_kernel, dim3(red, (unsigned)b.count), dim3(kBlock), 0, s, b, alpha, beta);
    GNNHIP_LAUNCH_CHECK("sgemm_tn_batch");
    return GNNHIP_OK;
}

int gemm_dispatch(int transA, int transB, int m, int n, int k, float alpha, const float* A, int lda,
                  const float* B, int ldb, float beta, float* C, int ldc, hipStream_t s)
{
    const bool wide_rows = k % 4 == 0 && lda % 4 == 0 && aligned16(A);
    if (!transA && n <= 4 && m >= 4096 && k >= 4 && (wide_rows || k <= 4 * kWave)) {
        switch (n) {
        case 1: launch_skinny<1>(transB, !wide_rows, m, k, alpha, A, lda, B, ldb, beta, C, ldc, s); break;
        case 2: launch_skinny<2>(transB, !wide_rows, m, k, alpha, A, lda, B, ldb, beta, C, ldc, s); break;
        case 3: launch_skinny<3>(transB, !wide_rows, m, k, alpha, A, lda, B, ldb, beta, C, ldc, s); break;
        default: launch_skinny<4>(transB, !wide_rows, m, k, alpha, A, lda, B, ldb, beta, C, ldc, s); break;
        }
        GNNHIP_LAUNCH_CHECK("sgemm_skinny");
        return GNNHIP_OK;
    }
    if (transA && !transB) return gemm_tn_batch_dispatch(1, &m, &n, &k, &A, &lda, &B, &ldb, alpha, beta, &C, &ldc, s);
    dim3 grid(ceil_div_u((size_t)m, BM), ceil_div_u((size_t)n, BN));
    dim3 block(kBlock);
    // few output tiles and a long k: split k so that about two workgroups per CU share the work
    int k_chunk = 0;
    float* partial = nullptr;
    const long long tiles = (long long)grid.x * grid.y;
    if (tiles <= kNumCU / 4 && k >= 256) {
        const long long chunk = splitk_chunk(tiles, k);
        const int splits = (int)(((long long)k + chunk - 1) / chunk);
        if (splits > 1) {
            void* q = nullptr;
            if (int rc = stream_scratch_slot(s, 2, sizeof(float) * (size_t)splits * m * n, &q)) return rc;
            partial = static_cast<float*>(q);
            k_chunk = (int)chunk;
            grid.z = splits;
        }
    }
    if (!transA && !transB)
        hipLaunchKernelGGL((sgemm_tile_kernel<false, false>), grid, block, 0, s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else if (!transA && transB)
        hipLaunchKernelGGL((sgemm_tile_kernel<false, true>), grid, block, 0, s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    else
        hipLaunchKernelGGL((sgemm_tile_kernel<true, true>), grid, block, 0, s, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, k_chunk, partial);
    if (partial) {
        const size_t total = (size_t)m * n;
        const unsigned rgrid = ceil_div_u(total, kWave) < 2048u ? ceil_div_u(total, kWave) : 2048u;
        hipLaunchKernelGGL(sgemm_splitk_reduce_kernel, dim3(rgrid), block, 0, s, m, n, (int)grid.z, alpha, partial, beta, C, ldc);
    }
    GNNHIP_LAUNCH_CHECK("sgemm_tile");
    return GNNHIP_OK;
}

}  // namespace gnnhip

using namespace gnnhip;

extern "C" int gnnhip_gemm_f32(int transA, int transB, int m, int n, int k, float alpha, const float* A, int lda,
                               const float* B, int ldb, float beta, float* C, int ldc, void* stream)
{
    GNNHIP_REQUIRE(m >= 0 && n >= 0 && k >= 0, "negative dimension in gemm (m=%d n=%d k=%d)", m, n, k);
    GNNHIP_REQUIRE((transA == 0 || transA == 1) && (transB == 0 || transB == 1), "trans flags must be 0 or 1");
    if (m == 0 || n == 0) return GNNHIP_OK;
    GNNHIP_REQUIRE(C != nullptr && ldc >= n, "bad output in gemm (ldc=%d n=%d)", ldc, n);
    if (k > 0) {
        GNNHIP_REQUIRE(A && B, "null operand in gemm");
        GNNHIP_REQUIRE(lda >= (transA ? m : k), "lda=%d too small", lda);
        GNNHIP_REQUIRE(ldb >= (transB ? k : n), "ldb=%d too small", ldb);
    }
    GNNHIP_REQUIRE(ceil_div_u((size_t)n, 64) <= 65535u, "n=%d too wide for the gemm grid", n);
    if (int rc = require_ready()) return rc;
    return gemm_dispatch(transA, transB, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, as_stream(stream));
}

extern "C" int gnnhip_gemm_tn_batch_f32(int count, const int* m, const int* n, const int* k, const float* const* A, const int* lda,
                                        const float* const* B, const int* ldb, float alpha, float beta, float* const* C, const int* ldc,
                                        void* stream)
{
    GNNHIP_REQUIRE(count >= 0, "negative count in gemm_tn_batch");
    if (count == 0) return GNNHIP_OK;
    GNNHIP_REQUIRE(m && n && k && A && lda && B && ldb && C && ldc, "null array in gemm_tn_batch");
    for (int p = 0; p < count; ++p) {
        GNNHIP_REQUIRE(m[p] >= 0 && n[p] >= 0 && k[p] >= 0, "negative dimension in gemm_tn_batch (product %d: m=%d n=%d k=%d)", p, m[p], n[p], k[p]);
        if (m[p] == 0 || n[p] == 0) continue;
        GNNHIP_REQUIRE(C[p] != nullptr && ldc[p] >= n[p], "bad output in gemm_tn_batch (product %d: ldc=%d n=%d)", p, ldc[p], n[p]);
        GNNHIP_REQUIRE(k[p] == 0 || (A[p] && B[p] && lda[p] >= m[p] && ldb[p] >= n[p]), "bad operand in gemm_tn_batch (product %d)", p);
        GNNHIP_REQUIRE(ceil_div_u((size_t)n[p], 64) <= 65535u, "n=%d too wide for the gemm grid", n[p]);
    }
    if (int rc = require_ready()) return rc;
    for (int at = 0; at < count; at += kGemmBatch) {
        const int take = count - at < kGemmBatch ? count - at : kGemmBatch;
        if (int rc = gemm_tn_batch_dispatch(take, m + at, n + at, k + at, A + at, lda + at, B + at, ldb + at, alpha, beta, C + at, ldc + at,
                                            as_stream(stream)))
            return rc;
    }
    return GNNHIP_OK;
}
