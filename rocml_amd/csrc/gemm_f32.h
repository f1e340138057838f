// 32-bit matrix products on the matrix cores: out[M,N] (+)= X[M,K] * W[N,K]^T with v_mfma_f32_16x16x4_f32, which multiplies
// and adds in full 32-bit precision (155 TFLOP/s from registers here; vector FMAs reach half of it).  Operands whose K and
// row strides are multiples of 4 and whose pointers are 16-byte aligned; everything else keeps the plain kernel.
//  * many rows: gemm_mfma_kernel with 32-bit elements (gemm_mfma.h): the same bytes a stage, 32 values of K instead of 64;
//  * up to 32 rows: gemm_f32_rows_kernel below.
// Measured against the plain kernel (microseconds, Qwen3-0.6B's layers): 1024 x 3072 into the stream 301 -> 11 at 4 rows and
// 446 -> 43 at 574, 4096 x 1024 122 -> 9 and 146 -> 59, the output matrix (151936 x 1024) 135 at 4 rows (4.6 TB/s); 2,048 rows
// run at 106 to 121 TFLOP/s.  The plain kernel's 64x64 blocks were a few dozen of 256 CUs, each a serial walk along K.
// Against 64 bits the sums are as close as before or closer (K is summed in 4 to 64 runs): 2.6e-7 for 9.6e-7 at 4 x 1024 x 3072.
// In both a lane reads four neighbouring K values of a row at once and hands them to four products one after the other,
// the same values of both operands each time: which of a product's K places a value takes does not matter to the sum.
#pragma once
#include "gemm_mfma.h"

// Up to 16 * RT rows, bound by the weights' bytes: a block owns 16 weight rows and all of K, its WAVES waves take turns
// along K in runs of 64 values (256 bytes of a row), read weights and activations straight into operand registers and meet
// once in LDS, in wave order: whole sums, no second kernel, any epilogue.  With k_piece < K a block has K only from
// blockIdx.y * k_piece on, and out is the workspace's [piece][M][N] (the caller instantiates the plain store).
template <int WAVES, int RT, int EPI>
__global__ void __launch_bounds__(64 * WAVES)
gemm_f32_rows_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ w, int ldw,
                     float* __restrict__ out, int ldo, int m, int n, int k, int k_piece) {
    __shared__ float red[WAVES][RT][16][17];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n0 = blockIdx.x * 16;
    const int part = (lane >> 4) * 4;
    x += blockIdx.y * k_piece;
    w += blockIdx.y * k_piece;
    out += (size_t)blockIdx.y * m * n;
    k = min(k - (int)blockIdx.y * k_piece, k_piece);
    // rows beyond M or N read the last one: they only feed sums that are not stored
    const float* wp = w + (size_t)min(n0 + (lane & 15), n - 1) * ldw + part;
    const float* xp[RT];
    f32x4_t acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        xp[r] = x + (size_t)min(r * 16 + (lane & 15), m - 1) * ldx + part;
        acc[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    int k0 = wave * 64;
#pragma unroll 2
    for (; k0 + 64 <= k; k0 += WAVES * 64) {
        f32x4_t a[4], b[RT][4];
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = *(const f32x4_t*)(wp + k0 + c * 16);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) b[r][c] = *(const f32x4_t*)(xp[r] + k0 + c * 16);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int r = 0; r < RT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][e], b[r][c][e], acc[r], 0, 0, 0);
    }
    // the rest of K, in the wave whose turn it is
    for (; k0 < k; k0 += 16) {
        const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
        const bool in = k0 + part < k;
        f32x4_t a = in ? *(const f32x4_t*)(wp + k0) : zero;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            f32x4_t b = in ? *(const f32x4_t*)(xp[r] + k0) : zero;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc[r], 0, 0, 0);
        }
        if ((k0 & 63) == 48) break;                   // (a run of 64 is one wave's)
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave][r][lane & 15][part + e] = acc[r][e];
    __syncthreads();
    constexpr int COLS = epi_gated(EPI) ? 8 : 16;
    for (int i = threadIdx.x; i < RT * 16 * COLS; i += 64 * WAVES) {
        int row = i / COLS, c = i % COLS;
        int col = n0 / 16 * COLS + c;
        if (row >= m || col >= (epi_gated(EPI) ? n / 2 : n)) continue;
        float* to = out + (size_t)row * ldo + col;
        float first = 0.f, second = 0.f;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) {
            first += red[v][row / 16][row % 16][epi_gated(EPI) ? 2 * c : c];
            if (epi_gated(EPI)) second += red[v][row / 16][row % 16][2 * c + 1];
        }
        if (epi_gated(EPI)) first = gated_mul<EPI>(first, second);
        *to = EPI == EPI_ACC ? *to + first : first;
    }
}

template <int EPI>
static int launch_f32_rows(const float* x, int ldx, const float* w, int ldw, float* out, int ldo, int m, int n, int k,
                           void* workspace, long long workspace_bytes, SplitPlan plan, hipStream_t stream) {
    const int blocks = ceil_div(n, 16), cus = cu_count();
    // A narrow product whose sums the next kernel adds up is cut along K as well while blocks are fewer than CUs (each
    // piece at least 512 of K): a CU pulls its weights at some 60 GB/s.  1024 x 3072 and 1024 x 2048 at 4 rows: 9.1 us
    // on average on 64 blocks, 5.5 on 256.
    int splits = 1;
    if (plan.defer && ldo == n && !epi_gated(EPI) && workspace)
        while (splits < 4 && splits * 2 <= plan.max_splits && blocks * splits * 2 <= cus && k / (splits * 2) >= 512 &&
               (long long)splits * 2 * m * n * 4 <= workspace_bytes)
            splits *= 2;
    const int k_piece = splits == 1 ? k : round_up(ceil_div(k, splits), 64);
    splits = ceil_div(k, k_piece);
    // waves a block: few blocks need many to have enough bytes on their way
    const int waves = k_piece > 512 && blocks * splits <= cus ? 16 : k_piece > 256 && blocks <= 4 * cus ? 8 : 4;
    const dim3 grid(blocks, splits);
#define F32_ROWS(W_, RT_)                                                                                                     \
    (splits > 1 ? gemm_f32_rows_kernel<W_, RT_, EPI_F32><<<grid, 64 * W_, 0, stream>>>(x, ldx, w, ldw, (float*)workspace, n, m, n, k, k_piece) \
                : gemm_f32_rows_kernel<W_, RT_, EPI><<<grid, 64 * W_, 0, stream>>>(x, ldx, w, ldw, out, ldo, m, n, k, k_piece))
    if (m <= 16) {
        if (waves == 16) F32_ROWS(16, 1);
        else if (waves == 8) F32_ROWS(8, 1);
        else F32_ROWS(4, 1);
    } else {
        if (waves == 16) F32_ROWS(16, 2);
        else if (waves == 8) F32_ROWS(8, 2);
        else F32_ROWS(4, 2);
    }
#undef F32_ROWS
    if (splits > 1) *plan.deferred = splits;
    return 0;
}

// Many rows: the ring kernel on 64x64 tiles (three blocks a CU) or 64x128, K cut in pieces (32-bit partial sums, as everywhere) where
// whole K leaves CUs idle.  Bound by the matrix cores: a stage (32 of K) is 1,024 clocks for a 64x64 tile, whatever else the CU holds.
// The constants of the estimate are a fit to 6,300 times of 1,105 products (33 to 1,500 rows, 18 outputs, K from 256 to 12288), 4 to
// 7 % off (root mean square); the choice by it is 1 % behind the best of both on average, 17 % at worst.
// Before the ring (operands staged through registers, 128x128 tiles beside 64x64), microseconds: 574 rows x 4096 x 1024 62 -> 52,
// gated 6144 x 1024 76 -> 67, 1024 x 3072 42 -> 37 with three pieces for six; 1000 x 4096 x 2048 146 -> 130.
using GemmTile64 = GemmTile<2, 2, 1, 1>;

template <int EPI>
static int launch_f32_tile(const float* x, int ldx, const float* w, int ldw, float* out, int ldo, int m, int n, int k,
                           void* workspace, long long workspace_bytes, SplitPlan plan, hipStream_t stream) {
    const int cus = cu_count();
    double best = 1e30;
    int wide = 64, splits = 1;
    for (int bn = 64; bn <= 128; bn += 64)
        for (int pieces = 1; pieces <= 8 && pieces <= plan.max_splits; ++pieces) {
            if (pieces > 1 && (epi_gated(EPI) || k / pieces < 128 || !workspace || (long long)pieces * m * n * 4 > workspace_bytes)) break;
            long long blocks = (long long)ceil_div(m, 64) * ceil_div(n, bn) * pieces;
            double stage = bn == 128 ? 1.042 : 0.538, fixed = bn == 128 ? 4.57 : 4.73;    // microseconds
            double t = (double)ceil_div(blocks, (long long)cus) * ceil_div(ceil_div(k, pieces), 32) * stage + fixed;
            if (pieces > 1) t += (double)pieces * m * n * 4.0 / 5.0e6 + (plan.defer && ldo == n ? 0.0 : 4.0);
            if (t < best) { best = t; wide = bn; splits = pieces; }
        }
    if (!rows_near(ldx, ldw, 4)) return launch_mfma_tile_as<EPI, GemmTile64, float>(x, ldx, w, ldw, out, ldo, m, n, k, splits, workspace, plan, stream);
    if (wide == 64) return launch_ring<EPI, RingTile<GemmTile64, 3>, float>(x, ldx, w, ldw, out, ldo, m, n, k, splits, workspace, plan, stream);
    return launch_ring<EPI, RingTile<GemmTile<2, 2, 1, 2>, 3>, float>(x, ldx, w, ldw, out, ldo, m, n, k, splits, workspace, plan, stream);
}
