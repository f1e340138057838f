// bfloat16 attention of long prompts over the paged cache, 64 query rows a wave: see attn_prompt_kernel.
#pragma once
#include "attention_mfma.h"

namespace prompt {

constexpr int ROWS = 64;                              // query rows of a wave, two tiles of 32
constexpr int SLOTS = 4;                              // pages of keys, and of values, in LDS
constexpr int TILE = 4 * ROWS;                        // query rows of a block
constexpr float MOST = 0x1p120f;                      // of a row's sum: its reciprocal is a number of all digits, too

template <int D>
struct Lds {
    static constexpr int PAGE = AM_PAGE * D * 2;      // bytes of a page's keys, and of its values
    static constexpr int PIECES = PAGE / 4096;        // loads of 1 KB a wave for one of them
    static constexpr int BYTES = 2 * SLOTS * PAGE;
};

typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

// 1 KB from memory to LDS at `lds`, 16 bytes a lane; a lane whose offset lies beyond the buffer leaves zeros.  Written as assembly
// because the compiler answers its own form of this load with a full wait before the next LDS read; it has no result register, and
// the kernel waits for it by count.
__device__ __forceinline__ void load_piece(i32x4_t buf, int lds, uint32_t offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(offset), "s"(buf) : "memory", "m0");
}

__device__ __forceinline__ i32x4_t buffer_of(const void* base, int bytes) {
    uint64_t a = (uint64_t)(uintptr_t)base;
    i32x4_t r = {(int)(uint32_t)a, (int)(uint32_t)(a >> 32), bytes, 0x00020000};
    return i32x4_t{__builtin_amdgcn_readfirstlane(r.x), __builtin_amdgcn_readfirstlane(r.y), r.z, r.w};
}

// The key whose scores are row i of the first product's 32: a lane's scores e are then keys 16 (e/8) + 8 (lane/32) + e%8, its
// probabilities the second product's operand and its values 16 consecutive bytes of a value row.
__device__ __forceinline__ int key_of_row(int i) { return (i & 16) | ((i & 4) << 1) | ((i & 8) >> 1) | (i & 3); }
// Where the 16-byte pieces of a row stand: piece p of a key row of 256 bytes at place p ^ (key % 16), of a value row of 128 bytes at
// p ^ (row / 2 % 8).  Sixteen lanes that read the same piece of sixteen rows then find every bank once.
__device__ __forceinline__ int key_place(int piece, int key) { return piece ^ (key & 15); }
__device__ __forceinline__ int value_place(int piece, int row) { return piece ^ (row >> 1 & 7); }

}  // namespace prompt

// What bounds prompt attention.  A product of 32 query rows with an operand of keys or values reads 1 KB of LDS for 32 clocks of its
// SIMD's matrix core, 128 bytes a clock and CU: all that LDS gives, before the pages' own way into it.  attn_prefill_mfma_kernel
// (32 rows a wave, pages through registers, two blocks a CU) reaches 0.95 PFLOP/s.  Here a wave has 64 rows and all 512 registers
// of its SIMD's lanes (128 of sums, 64 of queries, twice 32 of scores), so that an operand read once is multiplied twice:
//  * pages go from memory straight into swizzled LDS rows, asked for three and four visits before they are read; a barrier a page;
//  * nobody covers for a wave that waits, so its instructions are laid out one by one: behind each product two or three vector operations of
//    the softmax of the last 32 keys, operands read six pairs of products ahead, across steps and the page's barrier too;
//  * a row's reference stays what the maximum of its first page gave, so no step looks for a maximum, and none has a branch but the one that
//    hides keys on the diagonal.  Any reference gives the same quotient as long as the sums are numbers: probabilities, as bfloat16 and as
//    32-bit, have all their digits up to 2^127.  A wave with a row whose sums are not (scores some 80 above the first page's largest, or
//    something that is not finite) does its rows again at the end, with references that follow.  Heads whose queries and keys are normed
//    and have gains of one never come near it (|score| <= sqrt(128) = 11.3).
// Measured (32 query heads on 8; us, before and now): 8,192 tokens behind 24,576 others 4,038 and 3,108 (953 and 1,238 TFLOP/s), 8,192
// alone 626 and 496, four of 3,000 423 and 337; the rule in attention.hip has more.  The matrix cores are busy 59 % of the time at 1.95 GHz, where the chip's power
// holds the clock; the wave issues something 69 % of the time (5.4 vector operations a product) and waits for counters or the barrier 16 %.
// The error against 64 bits is that of the other kernel or a little less.  Measured and not kept: LDS reads with two lanes on a bank, the wait for
// all LDS reads before the barrier, operands four or seven pairs ahead, exponentials in equal parts behind both products of a pair: all
// equal (power); two waves for the halves of every page's keys with 128 rows a block: 3,417 where this takes 3,108, 28.0 at 1,024 tokens (30 and 37),
// 61 at 2,048; the compiler's own order of a step: 4,590; S in the vector registers (-amdgpu-mfma-vgpr-form): more moves, not fewer.
template <int D, bool QPREP>
__global__ void __launch_bounds__(AM_THREADS, 1)
attn_prompt_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out,
                   const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache,
                   const int* __restrict__ block_table, int bt_width,
                   const int* __restrict__ cu_seqlens, int n_seqs,
                   const int* __restrict__ token_pos, int hq, int hkv, float scale_log2e,
                   PrefillProj pj) {
    using namespace prompt;
    static_assert(D == 128, "the places of a row's pieces in LDS");
    using L = Lds<D>;
    constexpr int KK = D / 16, DT = D / 32, ROW = 2 * D;
    extern __shared__ uint4 am_smem[];
    const char* smem = (const char*)am_smem;
    const int smem_at = (int)(uintptr_t)(__attribute__((address_space(3))) void*)am_smem;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h2 = lane >> 5, col = lane & 31;
    // Heavy tiles first.  Blocks go to the dies in turn: a die gets neighbouring heads, which share their keys.
    const int total_tiles = gridDim.x / hq, in_tile = blockIdx.x % hq;
    const int h = hq % 8 == 0 ? in_tile % 8 * (hq / 8) + in_tile / 8 : in_tile, kvh = h / (hq / hkv);
    const AmTile at = am_find_tile<TILE>(cu_seqlens, n_seqs, total_tiles - 1 - (int)blockIdx.x / hq);
    if (at.b < 0) return;
    const int tile = at.tile, b = at.b, tok0 = at.tok0, n_new = at.n_new;
    const int* pages = block_table + (size_t)b * bt_width;
    const int pos0 = token_pos[tok0];
    const int row_lo = tile * TILE, row_hi = min(n_new, row_lo + TILE) - 1;
    const int w_lo = __builtin_amdgcn_readfirstlane(row_lo + wave * ROWS);
    const bool active = w_lo < n_new;
    const int w_hi = min(n_new - 1, w_lo + ROWS - 1);
    const int n_visits = (pos0 + row_hi) / AM_PAGE + 1;      // pages that the block's rows see keys of
    const int last = (pos0 + w_hi) / AM_PAGE;                // the last page that the wave's rows do

    // Pages on their way: keys four visits ahead, values three, their number counted by every wave.
    uint32_t koff[L::PIECES], voff[L::PIECES];
#pragma unroll
    for (int i = 0; i < L::PIECES; ++i) {
        int at = (wave * L::PIECES + i) * 1024 + lane * 16;
        int krow = at / ROW, kc = at % ROW / 16, vrow = at / 128, vc = at % 128 / 16;
        koff[i] = krow * ROW + key_place(kc, krow) * 16;
        voff[i] = vrow * 128 + value_place(vc, vrow) * 16;
    }
    typedef const __attribute__((address_space(4))) int* scalar_ptr_t;
    const scalar_ptr_t page_list = (scalar_ptr_t)(uintptr_t)pages;
    auto page_of = [&](int v) __attribute__((always_inline)) { return page_list[min(v, n_visits - 1)]; };
    auto page_buffer = [&](const bf16_t* cache, int id) __attribute__((always_inline)) {
        return buffer_of(cache + ((size_t)id * hkv + kvh) * AM_PAGE * D, L::PAGE);
    };
    auto request = [&](const bf16_t* cache, const uint32_t (&off)[L::PIECES], int v, int slot_at) __attribute__((always_inline)) {
        const i32x4_t buf = page_buffer(cache, page_of(v));
#pragma unroll
        for (int i = 0; i < L::PIECES; ++i)
            load_piece(buf, slot_at + (wave * L::PIECES + i) * 1024, v < n_visits ? off[i] : 0x80000000u);
    };
    int id3 = 0, id4 = 0;                              // the pages of the visits three and four ahead
    const int vbase = SLOTS * L::PAGE;

    bf16x8_t qf[2][KK];
    int my_pos[2];
    bool row_ok[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int my_row = w_lo + t * 32 + col;
        row_ok[t] = my_row < n_new;
        my_pos[t] = pos0 + my_row;
        const int token = tok0 + (row_ok[t] ? my_row : 0);
        if constexpr (QPREP) am_prepare_query<D>(pj, token, h, h2, row_ok[t], qf[t]);
        else am_load_query<D>(q + ((size_t)token * hq + h) * D, h2, row_ok[t], qf[t]);
    }

    float m[2] = {0.f, 0.f}, l[2] = {0.f, 0.f};
    f32x16_t o[2][DT], sc[2][2], zero;
    bf16x8_t pf[2][2];
#pragma unroll
    for (int e = 0; e < 16; ++e) zero[e] = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < DT; ++i) o[t][i] = zero;
    int kread[KK], vread[2];
#pragma unroll
    for (int i = 0; i < KK; ++i) kread[i] = key_of_row(col) * ROW + key_place(i * 2 + h2, key_of_row(col)) * 16;
#pragma unroll
    for (int u = 0; u < 2; ++u) vread[u] = col * 128 + value_place(u * 2 + h2, col) * 16;
    auto key_frag = [&](int slot, int half, int kk) __attribute__((always_inline)) {
        return __builtin_bit_cast(bf16x8_t, *(const u32x4_t*)(smem + slot * L::PAGE + kread[kk] + half * 32 * ROW));
    };
    auto value_frag = [&](int slot, int half, int u, int dt) __attribute__((always_inline)) {
        return __builtin_bit_cast(bf16x8_t, *(const u32x4_t*)(smem + vbase + slot * L::PAGE + (vread[u] ^ (half * 64)) + dt * 32 * 128));
    };
    auto scores = [&](int slot, int half, f32x16_t (&s)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            bf16x8_t kf = key_frag(slot, half, kk);
#pragma unroll
            for (int t = 0; t < 2; ++t) s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[t][kk], kk ? s[t] : zero, 0, 0, 0);
        }
    };
    auto add_values = [&](int slot, int half, const bf16x8_t (&p)[2][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                bf16x8_t vf = value_frag(slot, half, u, dt);
#pragma unroll
                for (int t = 0; t < 2; ++t) o[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, p[t][u], o[t][dt], 0, 0, 0);
            }
    };
    // exponentials of 16 scores: their sum, and the second product's operand
    auto exponentials = [&](const f32x16_t& s, float ref, bf16x8_t (&p)[2]) __attribute__((always_inline)) {
        float x[16], sum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            x[e] = fast_exp2(fmaf(s[e], scale_log2e, -ref));
            sum += x[e];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
            p[u] = __builtin_bit_cast(bf16x8_t, make_uint4(
                pack_bf16x2(x[8 * u + 0], x[8 * u + 1]), pack_bf16x2(x[8 * u + 2], x[8 * u + 3]),
                pack_bf16x2(x[8 * u + 4], x[8 * u + 5]), pack_bf16x2(x[8 * u + 6], x[8 * u + 7])));
        return sum;
    };
    // takes out the scores of keys behind their rows' positions
    auto hide = [&](int key0, f32x16_t (&s)[2]) __attribute__((always_inline)) {
        if (key0 + 31 <= pos0 + w_lo) return;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int key = key0 + 16 * (e >> 3) + 8 * h2 + (e & 7);
                s[t][e] = key <= my_pos[t] ? s[t][e] : -INFINITY;
            }
    };
    // Half way through visit v: the keys of v + 2 and the values of v + 1 are there, those of v and v - 1, which the visit's requests
    // overwrite, are read.  (What is being read at that time are the keys of v + 1 and the values of v.)
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * L::PIECES) : "memory");
    };
    i32x4_t kbuf, vbuf;
    auto aim = [&](int v) __attribute__((always_inline)) {
        kbuf = page_buffer(kcache, id4);
        vbuf = page_buffer(vcache, id3);
        id3 = id4;
        id4 = page_of(v + 5);
    };
    auto request_piece = [&](int v, int i) __attribute__((always_inline)) {       // the first PIECES are keys
        if (i < L::PIECES)
            load_piece(kbuf, smem_at + (v & 3) * L::PAGE + (wave * L::PIECES + i) * 1024, v + 4 < n_visits ? koff[i] : 0x80000000u);
        else
            load_piece(vbuf, smem_at + vbase + ((v + 3) & 3) * L::PAGE + (wave * L::PIECES + i - L::PIECES) * 1024,
                       v + 3 < n_visits ? voff[i - L::PIECES] : 0x80000000u);
    };
    // 32 keys that all rows see: their exponentials beside the next scores (keys of slot ks, half kh) and the products of the last
    // probabilities with their values (slot vs, half vh).  An operand is read AHEAD products' pairs before its products, the first ones by the step
    // before (ks2 ... vh2: the next step's).  The rows' references stay as they are.
    constexpr int PAIRS = KK + 2 * DT, RING = 8, AHEAD = 6;
    static_assert(KK == 2 * DT && PAIRS % RING == 0, "scores and values in turn");
    bf16x8_t ring[RING];
    auto operand = [&](int j, int ks, int kh, int vs, int vh) __attribute__((always_inline)) {
        return j & 1 ? value_frag(vs, vh, (j >> 1) / DT, (j >> 1) % DT) : key_frag(ks, kh, j >> 1);
    };
    auto step = [&](f32x16_t (&s)[2], f32x16_t (&next)[2], int ks, int kh, int vs, int vh, int ks2, int kh2, int vs2, int vh2,
                    auto between) __attribute__((always_inline)) {
        uint32_t pn[2][8];
        float sum[2] = {0.f, 0.f}, x[2] = {0.f, 0.f};
        auto finish = [&](int j) __attribute__((always_inline)) {
            sum[j >> 3] += x[0];
            sum[j >> 3] += x[1];
            pn[j >> 3][j & 7] = pack_bf16x2(x[0], x[1]);
            asm volatile("" : "+v"(sum[j >> 3]), "+v"(pn[j >> 3][j & 7]));
        };
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < PAIRS; ++j) {
            const int to = j + AHEAD;
            ring[to % RING] = to < PAIRS ? operand(to, ks, kh, vs, vh) : operand(to - PAIRS, ks2, kh2, vs2, vh2);
            const int i = j >> 1;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (j & 1) o[t][i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[j % RING], pf[t][i / DT], o[t][i % DT], 0, 0, 0);
                else next[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[j % RING], qf[t][i], i ? next[t] : zero, 0, 0, 0);
                if (t == 0) {
                    if (j) finish(j - 1);
                    between(j);
                } else {
                    const int e = 2 * (j & 7), row = j >> 3;
                    if (e == 0) asm volatile("" : "+a"(s[row]));
                    x[0] = fast_exp2(fmaf(s[row][e], scale_log2e, -m[row]));
                    x[1] = fast_exp2(fmaf(s[row][e + 1], scale_log2e, -m[row]));
                    asm volatile("" : "+v"(x[0]), "+v"(x[1]));      // (not later)
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        finish(PAIRS - 1);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            l[t] += sum[t];
#pragma unroll
            for (int u = 0; u < 2; ++u) pf[t][u] = __builtin_bit_cast(bf16x8_t, make_uint4(pn[t][4 * u], pn[t][4 * u + 1], pn[t][4 * u + 2], pn[t][4 * u + 3]));
        }
    };
    auto pass_by = [&](int v) __attribute__((always_inline)) {
        meet();
        aim(v);
#pragma unroll
        for (int i = 0; i < 2 * L::PIECES; ++i) request_piece(v, i);
    };
    request(kcache, koff, 0, smem_at);
    request(kcache, koff, 1, smem_at + L::PAGE);
    request(vcache, voff, 0, smem_at + vbase);
    request(kcache, koff, 2, smem_at + 2 * L::PAGE);
    request(vcache, voff, 1, smem_at + vbase + L::PAGE);
    request(kcache, koff, 3, smem_at + 3 * L::PAGE);
    request(vcache, voff, 2, smem_at + vbase + 2 * L::PAGE);
    id3 = page_of(3);
    id4 = page_of(4);
    int v = 0;
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(4 * L::PIECES) : "memory");
    if (active) {
        // the first page's maxima are the references (every row sees its first key)
        scores(v & 3, 0, sc[0]);
        scores(v & 3, 1, sc[1]);
        hide(0, sc[0]);
        hide(32, sc[1]);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 16; ++e) mx = fmaxf(fmaxf(mx, sc[0][t][e]), sc[1][t][e]);
            m[t] = max_across_halves(mx) * scale_log2e;
            l[t] = exponentials(sc[0][t], m[t], pf[t]);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) ring[j] = operand(j, (v + 1) & 3, 0, v & 3, 0);
        __builtin_amdgcn_s_waitcnt(0x0f70);            // (vmcnt(0): the compiler waits for nothing of its own in the loop)
        for (; v < last; ++v) {
            const int here = v & 3, after = (v + 1) & 3, behind = (v + 2) & 3;
            meet();
            aim(v);
            step(sc[1], sc[0], after, 0, here, 0, after, 1, here, 1, [&](int j) __attribute__((always_inline)) {
                if (j % 2 == 0 && j / 2 < 2 * L::PIECES) request_piece(v, j / 2);
            });
            hide((v + 1) * AM_PAGE, sc[0]);
            step(sc[0], sc[1], after, 1, here, 1, behind, 0, after, 0, [&](int) __attribute__((always_inline)) {});
            hide((v + 1) * AM_PAGE + 32, sc[1]);
        }
        pass_by(v);
        add_values(v & 3, 0, pf);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            l[t] += exponentials(sc[1][t], m[t], pf[t]);
        }
        add_values(v & 3, 1, pf);
        ++v;
    }
    for (; v < n_visits; ++v) pass_by(v);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // no load is on its way into LDS when the block ends
#pragma unroll
    for (int t = 0; t < 2; ++t) l[t] = sum_across_halves(l[t]);
    if (!active) return;
    // Where a reference was too far from its row's maximum, or something is no finite number, the wave does its rows again: 32 keys at a
    // time straight from memory, with references that follow.  Where all rows do (8,192 tokens, 32 heads, scores some 130 apart) the
    // kernel takes 1,500 us (without it 489, attn_prefill_mfma_kernel 600); each of the wave's two tiles by itself 2,290, the
    // next keys asked for ahead 1,520, references that follow inside the first pass 10 % more for all others.
    bool bad = false;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        float finite = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) finite = fmaf(o[t][dt][e], 0.f, finite);
        bad |= row_ok[t] && !(l[t] > 0.f && l[t] < MOST && finite == 0.f);
    }
    if (__builtin_amdgcn_ballot_w64(bad)) {
        int hi[2];                                      // the last key that a tile's rows see, -1: it has no rows
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            m[t] = -INFINITY;
            l[t] = 0.f;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[t][dt] = zero;
            hi[t] = w_lo + t * 32 < n_new ? pos0 + min(n_new - 1, w_lo + t * 32 + 31) : -1;
        }
#pragma unroll 1
        for (int key0 = 0; key0 <= max(hi[0], hi[1]); key0 += 32) {
            const size_t page = (size_t)pages[key0 / AM_PAGE] * hkv + kvh;
            const bf16_t* krow = kcache + (page * AM_PAGE + key0 % AM_PAGE + key_of_row(col)) * D + h2 * 8;
            const bf16_t* vrow = vcache + (page * D + col) * AM_PAGE + key0 % AM_PAGE + h2 * 8;
            bf16x8_t kf[KK], vf[DT][2];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) kf[kk] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(krow + kk * 16));
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int u = 0; u < 2; ++u) vf[dt][u] = __builtin_bit_cast(bf16x8_t, *(const uint4*)(vrow + dt * 32 * AM_PAGE + u * 16));
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (key0 > hi[t]) continue;             // (what is not finite there is none of these rows')
                f32x16_t s = zero;
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kk], qf[t][kk], s, 0, 0, 0);
                float mx = -INFINITY;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int key = key0 + 16 * (e >> 3) + 8 * h2 + (e & 7);
                    s[e] = row_ok[t] && key <= my_pos[t] ? s[e] : -INFINITY;
                    mx = fmaxf(mx, s[e]);
                }
                const float m_new = fmaxf(m[t], max_across_halves(mx) * scale_log2e), ref = m_new == -INFINITY ? 0.f : m_new;
                const float corr = fast_exp2(m[t] - ref);
                m[t] = m_new;
                l[t] = l[t] * corr + exponentials(s, ref, pf[t]);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[t][dt][e] *= corr;
#pragma unroll
                    for (int u = 0; u < 2; ++u) o[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt][u], pf[t][u], o[t][dt], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) l[t] = sum_across_halves(l[t]);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        if (!row_ok[t]) continue;
        const float inv = 1.0f / l[t];
        bf16_t* orow = out + ((size_t)(tok0 + w_lo + t * 32 + col) * hq + h) * D;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                uint2 v = make_uint2(pack_bf16x2(o[t][dt][4 * e4] * inv, o[t][dt][4 * e4 + 1] * inv),
                                     pack_bf16x2(o[t][dt][4 * e4 + 2] * inv, o[t][dt][4 * e4 + 3] * inv));
                *(uint2*)(orow + dt * 32 + 8 * e4 + 4 * h2) = v;
            }
    }
}
