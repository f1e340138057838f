// The many-rows product of launches that leave a CU one or two small tiles: see gemm_ring_kernel.
#pragma once
#include "gemm_pingpong.h"

// A tile with a ring of STAGES stages in LDS.
template <typename T, int STAGES>
struct RingTile : T {
    static constexpr int S = STAGES, ROW = 128, STAGE = (T::BM + T::BN) * ROW, LDS_BYTES = S * STAGE;
    static_assert(LDS_BYTES <= 160 * 1024 && S >= 3, "stages fit the LDS");
};

template <int SET> struct RingSet { static constexpr int value = SET; };

// Products of which a CU gets one or two tiles: prompts of a few hundred tokens, few rows with K in pieces, weights from memory.
// What bounds them: with operands staged through registers a block had one stage on its way, so a 128x128 tile's stage of 64 took
// 0.58 us where its products need 0.22: a trip to memory.  Here S stages of operands go straight into LDS (no registers, unpadded
// rows whose 16-byte pieces are XOR-swizzled by the row), S - 1 of them on their way while one is multiplied.  A stage's operands
// are read into a second set of registers between the products of the stage before, so a wave has products to issue right behind
// the one barrier of a stage, and that barrier is also what gives the stage's place back to the loads.
// Now the L2s bound it where all CUs pull: 32 KB a stage and CU at 14 TB/s, 0.58 us with all 256 CUs (128x128 tiles, K of 4096),
// 0.37 with a few; without the loads 0.39, without the LDS reads 0.56.  Five stages for four, reads in the first five eighths of a
// stage, eight waves for four: equal.  Rows padded in memory: equal (the L2's channels are hashed).
// Against the kernels it replaced (registers, double-buffered LDS; microseconds): 670 rows x 4096 x 1024 16.5 -> 12.2, gated 6144 x
// 1024 19.6 -> 16.4, 1024 x 3072 13.7 in four pieces -> 10.6 in two; 64 rows x 4096 x 12288 29 in eight pieces -> 22.5 in four,
// 6144 x 4096 16.7 -> 13.6; 512 rows x 6144 x 4096 40 -> 33.  Over 2,454 whole and gated products of 17 to 3,000 rows 0.81 of the time
// (geometric mean; 65 to 256 gated rows 0.58), one in thirty or so more than 3 % slower and six more than 10 %: wide outputs at 40 to 128 rows,
// whose blocks were two a CU (128 x 151936 x 1024 90 -> 97, 43 x 32768 x 2048 29 -> 32).  32-bit: 0.92 of the time over 400.
// Sums are formed in the order of gemm_mfma_kernel's (the same bits); in 32 bits in runs of 512 of K.
template <int EPI, typename T, typename E = bf16_t>
__global__ void __launch_bounds__(T::THREADS, 2)
gemm_ring_kernel(const E* __restrict__ x, int ldx, const E* __restrict__ w, int ldw,
                 void* __restrict__ out, int ldo, int m, int n, int k, int tiles_m, int n_tiles,
                 int k_per_split, long long split_stride) {
    extern __shared__ u32x4_t gm_smem[];              // [S stages][rows of x, rows of w][128 bytes, in swizzled pieces]
    using pingpong::i32x4_t;
    constexpr int MT = T::MT, NT = T::NT, S = T::S, LOADS = T::PA + T::PB, SIZE = sizeof(E), PIECE = 16 / SIZE, BK = 8 * PIECE;
    constexpr int DEAL = tile_deal<EPI, T, E>();
    const int smem = (int)(uintptr_t)(__attribute__((address_space(3))) void*)gm_smem;
    int per_xcd = gridDim.x / 8;
    int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    int split = logical / n_tiles;
    logical -= split * n_tiles;
    const int ks = split * k_per_split;
    if (ks >= k) return;
    k = min(k - ks, k_per_split);
    out = (float*)out + split * split_stride;
    int band_tiles = GM_BAND * (n_tiles / tiles_m), band = logical / band_tiles, in_band = logical - band * band_tiles;
    int band_rows = min(GM_BAND, tiles_m - band * GM_BAND);
    const int m0 = (band * GM_BAND + in_band % band_rows) * T::BM, n0 = (in_band / band_rows) * T::BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / T::WAVES_N, wn = wave % T::WAVES_N;
    const int nk = (k + BK - 1) / BK;

    // A stage's rows in runs of eight, dealt to the waves; a lane's place of a run holds piece (place ^ row) of its row.
    const int rows_x = min(m - m0, T::BM), rows_w = min(n - n0, T::BN);
    const i32x4_t xbuf = pingpong::buffer_of(x + (size_t)m0 * ldx + ks, ((long long)(rows_x - 1) * ldx + k) * SIZE);
    const i32x4_t wbuf = pingpong::buffer_of(w + (size_t)n0 * ldw + ks, ((long long)(rows_w - 1) * ldw + k) * SIZE);
    const int chunk = ((lane & 7) ^ (lane >> 3)) * PIECE;
    uint32_t off[LOADS];
#pragma unroll
    for (int r = 0; r < LOADS; ++r) {
        const bool is_w = r >= T::PA;
        int row = ((is_w ? r - T::PA : r) * (T::THREADS / 64) + wave) * 8 + (lane >> 3);
        if (is_w) {                                   // the weight row whose place this is (tile_lds_row, the other way)
            int in = row % (16 * DEAL);
            row = row - in + in % 16 / 4 * (4 * DEAL) + in / 16 * 4 + in % 4;
        }
        row = min(row, (is_w ? rows_w : rows_x) - 1);
        off[r] = ((uint32_t)row * (uint32_t)(is_w ? ldw : ldx) + chunk) * SIZE;
    }
    int kt_load = 0, slot_load = 0;
    auto request = [&](int r) {                       // run r of stage kt_load
        const bool is_w = r >= T::PA;
        const int to = smem + slot_load * T::STAGE + ((is_w ? T::BM : 0) + ((is_w ? r - T::PA : r) * (T::THREADS / 64) + wave) * 8) * T::ROW;
        pingpong::load_rows(is_w ? wbuf : xbuf, to, kt_load * BK + chunk < k ? off[r] + (uint32_t)kt_load * 128u : pingpong::NOWHERE);
    };
    auto next_request = [&]() {
        ++kt_load;
        slot_load = slot_load + 1 == S ? 0 : slot_load + 1;
    };
    const char* base = (const char*)gm_smem;
    const int swz = ((lane >> 4) ^ (lane & 7)) * 16;
    const int fa = (wm * MT * 16 + (lane & 15)) * T::ROW + swz, fb = (T::BM + wn * NT * 16 + (lane & 15)) * T::ROW + swz;
    u32x4_t a[2][2][MT], b[2][2][NT];
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // operand piece p of a stage into set `set`
    auto read = [&](int set, const char* from, int p) {
        const int s = p / (MT + NT), q = p % (MT + NT);
        if (q < MT) a[set][s][q] = *(const u32x4_t*)(from + (fa ^ (s * 64)) + q * 16 * T::ROW);
        else b[set][s][q - MT] = *(const u32x4_t*)(from + (fb ^ (s * 64)) + (q - MT) * 16 * T::ROW);
    };
    constexpr int READS = 2 * (MT + NT), PRODUCTS = 2 * MT * NT;
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int r = 0; r < LOADS; ++r) request(r);
        next_request();
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 1) * LOADS) : "memory");
#pragma unroll
    for (int p = 0; p < READS; ++p) read(0, base, p);
    int slot = 0;
    auto stage = [&](auto set_) {
        constexpr int SET = decltype(set_)::value;
        // the next stage is there, and every wave has this one in registers: its place is asked for again
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * LOADS) : "memory");
        slot = slot + 1 == S ? 0 : slot + 1;
        const char* from = base + slot * T::STAGE;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < PRODUCTS; ++p) {
#pragma unroll
            for (int r = p * READS / PRODUCTS; r < (p + 1) * READS / PRODUCTS; ++r) read(SET ^ 1, from, r);
#pragma unroll
            for (int r = p * LOADS / PRODUCTS; r < (p + 1) * LOADS / PRODUCTS; ++r) request(r);
            const int s = p / (MT * NT), i = p / NT % MT, j = p % NT;
            if constexpr (SIZE == 2) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag4(b[SET][s][j]), as_frag4(a[SET][s][i]), acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b[SET][s][j][e]), __uint_as_float(a[SET][s][i][e]), acc[i][j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        next_request();
    };
    // 32-bit operands: sums of 512 of K each, added up, so that a long K is as close to the exact sums as K in pieces would be
    f32x4_t total[SIZE == 4 ? MT : 1][NT];
    if constexpr (SIZE == 4) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) total[i][j] = acc[i][j];
    }
    auto add_up = [&]() {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                total[i][j] += acc[i][j];
                acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
    };
    for (int kt = 0; kt + 1 < nk; kt += 2) {
        stage(RingSet<0>{});
        stage(RingSet<1>{});
        if constexpr (SIZE == 4) {
            if ((kt & 14) == 14) add_up();
        }
    }
    if (nk & 1) stage(RingSet<0>{});
    if constexpr (SIZE == 4) {
        add_up();
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load is on its way into LDS when the block ends
    tile_epilogue<EPI, T, E>(acc, out, ldo, m, n, m0, n0, wm, wn, lane);
}
