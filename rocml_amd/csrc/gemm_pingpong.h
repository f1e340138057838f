// The many-rows product on 256x256 tiles, operands straight from memory into LDS and the two waves of a SIMD in opposite
// phases: see gemm_pingpong_kernel.
#pragma once
#include "gemm_mfma.h"

namespace pingpong {

using Tile = GemmTile256;                             // eight waves of 128x64: the epilogue's layout
constexpr int ROW = GM_BK * 2;                        // bytes of an LDS row: 64 K values, unpadded
constexpr int SIDE = 256 * ROW, STAGE = 2 * SIDE;     // one operand's rows, both
constexpr int LDS_BYTES = 2 * STAGE;

typedef __attribute__((ext_vector_type(4))) int i32x4_t;

// 1 KB (eight rows of a stage) from memory to LDS at `lds`; a lane whose offset lies beyond the buffer leaves zeros.
// Written as assembly because the compiler answers its own form of this load with a full wait before the next LDS read;
// it has no result register, and the kernel waits for it by count.
__device__ __forceinline__ void load_rows(i32x4_t buf, int lds, uint32_t offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(offset), "s"(buf) : "memory", "m0");
}

__device__ __forceinline__ i32x4_t buffer_of(const void* base, long long bytes) {
    uint64_t a = (uint64_t)(uintptr_t)base;
    i32x4_t r = {(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)min(bytes, (long long)0x7fffffff), 0x00020000};
    return i32x4_t{__builtin_amdgcn_readfirstlane(r.x), __builtin_amdgcn_readfirstlane(r.y), __builtin_amdgcn_readfirstlane(r.z), r.w};
}

constexpr uint32_t NOWHERE = 0x80000000u;             // an offset beyond every buffer

}  // namespace pingpong

// What bounds the 256x256 product: a 64-wide stage is 2,048 clocks of the matrix cores, and the LDS moves 192 KB of reads
// and 64 KB of arrivals for it, 2,048 clocks of its own; the clock is held near 1.9 GHz by the chip's power.  So neither
// unit may wait for the other, and no wave may spend issue slots on moving operands through registers:
//  * a stage goes from memory into unpadded, XOR-swizzled LDS rows without passing registers, in four parts of 16 KB, seven
//    phases before it is read: each part's place is asked for again one phase after its last reader has met the others;
//  * a stage is four phases of 16 products a wave (half of its rows by half of its columns, all 64 of K).  The two waves of
//    a SIMD (one from each half of the block) are one step apart: while one issues its products, the other reads the
//    operands of its next phase and asks for a part of a later stage; a barrier after every step keeps them apart.  The
//    reads of a phase are 8, 4, 8 and 4 pieces of 1 KB;
//  * a block a CU walks through its share of the tiles, and the parts of the next tile are asked for during the last two
//    stages of this one, so that they arrive while the sums are written.
// Measured (random operands; the kernel it replaced staged through registers with 32x32x16 products, one barrier a stage):
// 8192 x 24576 x 4096 gated 1,370 -> 1,161 us (1.20 -> 1.42 PFLOP/s), 8192 x 4096 x 12288 into the stream 765 -> 584,
// 2048 x 24576 x 4096 gated 352 -> 287, 2048 x 6144 x 4096 94.7 -> 85 (launched one after another on one machine; the
// gated one took 1,095 and 1,132 on others, and 5 % less with a silu of less than whole 32-bit precision).  A stage takes 2,519 clocks at 1.9 GHz; without the loads
// 2,200 at 2.05, without the LDS reads 2,230, without both 2,160 at 2.2 (2.0 PFLOP/s): what is left is power and the
// arrivals' share of the LDS.  Not kept: a ring of five half stages (all 160 KB of LDS, nine phases ahead): 2 % slower; six
// reads in every phase instead of 8, 4, 8, 4: equal; without the raised priority around the products: equal.
// Sums are formed in the order of gemm_mfma_kernel's: the results are the same bits.
template <int EPI>
__global__ void __launch_bounds__(512, 2)
gemm_pingpong_kernel(const bf16_t* __restrict__ x, int ldx, const bf16_t* __restrict__ w, int ldw,
                     void* __restrict__ out, int ldo, int m, int n, int k, int tiles_m, int n_tiles,
                     int k_per_split, long long split_stride, int items) {
    using namespace pingpong;
    using T = Tile;
    extern __shared__ u32x4_t gm_smem[];
    const int smem = (int)(uintptr_t)(__attribute__((address_space(3))) void*)gm_smem;
    constexpr int DEAL = tile_deal<EPI, T>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    // Of the work items (tiles times K pieces) an XCD has a run of neighbours, of which each of its blocks takes every
    // gridDim.x / 8 th one.
    const int per_xcd = (items + 7) / 8, blocks = gridDim.x / 8;
    const int last = min(((int)blockIdx.x % 8 + 1) * per_xcd, items);
    struct Item { int split, m0, n0, ks, k; };
    auto item_of = [&](int index) {
        Item t;
        t.split = index / n_tiles;
        int tile = index - t.split * n_tiles;
        int band_tiles = GM_BAND * (n_tiles / tiles_m), band = tile / band_tiles, in_band = tile - band * band_tiles;
        int band_rows = min(GM_BAND, tiles_m - band * GM_BAND);
        t.m0 = (band * GM_BAND + in_band % band_rows) * T::BM;
        t.n0 = (in_band / band_rows) * T::BN;
        t.ks = t.split * k_per_split;
        t.k = min(k - t.ks, k_per_split);
        return t;
    };
    int index = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (index >= last) return;

    // A stage arrives in four parts of 128 rows, in the order the phases read them: half 0 of every wave's weight columns,
    // half 0 of its rows of x, half 1 of the columns, half 1 of the rows.  Of every part a wave loads two runs of eight
    // rows.  The stages of one item follow those of the one before it, two stages ahead of the products.
    const int xrow = wm * 128 + wn * 16, wrow = (wave >> 1) * 64 + (wave & 1) * 16;
    const int chunk = ((lane & 7) ^ (lane >> 3)) * 8; // the row's piece that this lane's place holds (rows p, p + 8, ... alike)
    uint32_t off[4][2];
    i32x4_t xbuf, wbuf;
    int load_index = index, load_k = 0, kt_load = 0, slot_load = 0;
    auto aim = [&]() {                                // at the first stage of item load_index, or at nothing
        if (load_index >= last) {
            load_k = 0;                               // every piece lies beyond K: zeros, no traffic
            return;
        }
        Item t = item_of(load_index);
        load_k = t.k;
        const int rows_x = min(m - t.m0, 256), rows_w = min(n - t.n0, 256);
        xbuf = buffer_of(x + (size_t)t.m0 * ldx + t.ks, ((long long)(rows_x - 1) * ldx + t.k) * 2);
        wbuf = buffer_of(w + (size_t)t.n0 * ldw + t.ks, ((long long)(rows_w - 1) * ldw + t.k) * 2);
#pragma unroll
        for (int part = 0; part < 4; ++part)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                bool is_w = !(part & 1);
                int half = part >> 1;
                int row = (is_w ? wrow + half * 32 : xrow + half * 64) + u * 8 + (lane >> 3);
                if (is_w) {                           // the weight row whose place this is (tile_lds_row, the other way)
                    int in = row % (16 * DEAL);
                    row = row - in + in % 16 / 4 * (4 * DEAL) + in / 16 * 4 + in % 4;
                }
                row = min(row, (is_w ? rows_w : rows_x) - 1);
                off[part][u] = ((uint32_t)row * (uint32_t)(is_w ? ldw : ldx) + chunk) * 2u;
            }
    };
    auto request = [&](int part) {
        bool in = kt_load * GM_BK + chunk < load_k;
        uint32_t at = (uint32_t)kt_load * (GM_BK * 2);
        int to = smem + slot_load * STAGE + (part & 1 ? xrow + (part >> 1) * 64 : 256 + wrow + (part >> 1) * 32) * ROW;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            load_rows(part & 1 ? xbuf : wbuf, to + u * 8 * ROW, in ? off[part][u] + at : NOWHERE);
        if (part == 3) {
            slot_load ^= 1;
            if (++kt_load * GM_BK >= load_k) {
                load_index += blocks;
                kt_load = 0;
                aim();
            }
        }
    };
    const char* base = (const char*)gm_smem;
    const int swz = ((lane >> 4) ^ (lane & 7)) * 16;  // slice 0's piece of a row; slice 1's is 64 bytes across (bit 2 of the piece)
    const int fa = (wm * 128 + (lane & 15)) * ROW + swz, fb = SIDE + (wn * 64 + (lane & 15)) * ROW + swz;
    bf16x8_t a[2][4], b0[2][2], b1[2][2];
    f32x4_t acc[T::MT][T::NT];
    int slot = 0;                                     // the stage's half of LDS

#define PP_READ_A(slot_, half_)                                                                                          \
    _Pragma("unroll") for (int s = 0; s < 2; ++s) _Pragma("unroll") for (int i = 0; i < 4; ++i)                         \
        a[s][i] = as_frag4(*(const u32x4_t*)(base + (slot_) * STAGE + (fa ^ (s * 64)) + ((half_)*4 + i) * 16 * ROW));
#define PP_READ_B(slot_, half_, b_)                                                                                      \
    _Pragma("unroll") for (int s = 0; s < 2; ++s) _Pragma("unroll") for (int j = 0; j < 2; ++j)                         \
        b_[s][j] = as_frag4(*(const u32x4_t*)(base + (slot_) * STAGE + (fb ^ (s * 64)) + ((half_)*2 + j) * 16 * ROW));
#define PP_MEET() asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)\n\ts_barrier" ::: "memory")
#define PP_PRODUCTS(ha_, hb_, b_)                                                                                      \
    __builtin_amdgcn_sched_barrier(0);                                                                                 \
    __builtin_amdgcn_s_setprio(1);                                                                                     \
    _Pragma("unroll") for (int s = 0; s < 2; ++s) _Pragma("unroll") for (int i = 0; i < 4; ++i)                         \
        _Pragma("unroll") for (int j = 0; j < 2; ++j) acc[(ha_)*4 + i][(hb_)*2 + j] =                                  \
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(b_[s][j], a[s][i], acc[(ha_)*4 + i][(hb_)*2 + j], 0, 0, 0);         \
    __builtin_amdgcn_s_setprio(0);                                                                                     \
    __builtin_amdgcn_sched_barrier(0);                                                                                 \
    asm volatile("s_barrier" ::: "memory");

    aim();
#pragma unroll
    for (int i = 0; i < 8; ++i) request(i & 3);
    PP_MEET();
    PP_READ_B(0, 0, b0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (; index < last; index += blocks) {
        const Item item = item_of(index);
        const int nk = (item.k + GM_BK - 1) / GM_BK;
#pragma unroll
        for (int i = 0; i < T::MT; ++i)
#pragma unroll
            for (int j = 0; j < T::NT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (wm) asm volatile("s_barrier" ::: "memory");
        for (int kt = 0; kt < nk; ++kt) {
            PP_READ_A(slot, 0);
            request(0);
            PP_MEET();
            PP_PRODUCTS(0, 0, b0);
            PP_READ_B(slot, 1, b1);
            request(1);
            PP_MEET();
            PP_PRODUCTS(0, 1, b1);
            PP_READ_A(slot, 1);
            request(2);
            PP_MEET();
            PP_PRODUCTS(1, 0, b0);
            slot ^= 1;
            PP_READ_B(slot, 0, b0);
            request(3);
            PP_MEET();
            PP_PRODUCTS(1, 1, b1);
        }
        if (!wm) asm volatile("s_barrier" ::: "memory");
        tile_epilogue<EPI, T>(acc, (float*)out + item.split * split_stride, ldo, m, n, item.m0, item.n0, wm, wn, lane);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load is on its way into LDS when the block ends
#undef PP_READ_A
#undef PP_READ_B
#undef PP_MEET
#undef PP_PRODUCTS
}
