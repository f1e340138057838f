// bfloat16 attention over a cache of latent rows on the gfx950 matrix cores.
//
// The cache holds one row of DK numbers per position, [page, 64, DK]; all query heads share it (one
// key/value "head"), a key is the whole row and its value is the row's first DV numbers.  A layer
// whose keys and values are expanded from a latent vector reaches this form by folding the key
// expansion into its queries and the value expansion into a product behind the attention.
//
// Rows of work are the (token, head) pairs of a step: the queries [T, H, DK] and the outputs
// [T, H, DV] are plain matrices of T * H rows, and row r of a sequence's new tokens stands at
// position pos0 + r / H.  A block takes 64 RT consecutive rows of one sequence (RT tiles of 16 per
// wave: the 16 columns of an MFMA; RT = 2 for prompts, where every key operand read from LDS then
// feeds two products and a loaded key serves 128 rows, RT = 1 for the few rows of a decode step and
// for the widest sizes, whose two tiles of outputs and queries would not fit a lane's 512 registers)
// and one split of their keys; keys come 32 at a time through LDS, once as
// rows (the first product, S^T = K Q^T, reads 8 numbers of a key per lane) and once transposed
// (the second, O^T = V^T P^T, reads 8 keys of a number per lane): the transposition happens on
// the way into LDS, the cache keeps the rows only.  With many rows per sequence (a prompt) the
// 64 rows share every key they load; with few (a decode step: H rows per sequence) the key range
// is cut into splits whose partial results a second kernel merges by log-sum-exp, in split order.
//
// Online softmax per column as in attention_mfma.h; scores scaled after the dot product, base-2
// exponentials.  A window limits the keys of a row to (pos - window, pos].
// KD: 32-number steps of the first product (DK <= 32 KD), DT: 16-number tiles of the output
// (DV <= 16 DT); numbers beyond DK or DV are zeros in LDS and in the query operand.
#pragma once
#include "attention_mfma.h"

constexpr int AL_ROWS = 64;           // rows of a block
constexpr int AL_KEYS = 32;           // keys of a piece
constexpr int AL_VROW = AL_KEYS + 8;  // bf16 per row of the transposed piece (16 bytes of padding)
constexpr float AL_LAZY_MAX = 8.0f;   // how far a row's maximum may run ahead of its exponents' reference (powers of two)

// Where the transposed piece keeps number d of the keys (bf16 units): rows of AL_VROW and 32 more
// after every eight rows, so that rows eight apart, which neighbouring groups of lanes write at
// the same time, lie 16 banks apart.
__device__ __forceinline__ int al_vrow_at(int d) { return d * AL_VROW + (d >> 3) * 32; }

// Keys as rows: the first product's tile u reads key 8 (c / 4) + 4 u + c % 4 in lane column c; that key
// is stored at row 16 u + c, so the 16 lanes of a tile read 16 consecutive rows.  A thread that
// stages the piece takes the two keys of one column c (they are 4 apart) and writes rows c and
// 16 + c: 16 neighbouring lanes write 16 consecutive rows.  In the transposed copy the two keys
// stand side by side (key 8 G + 4 u + i at place 8 G + 2 i + u of its row), one 4-byte store; the
// probabilities are packed in the same order.

template <int KD, int DT>
struct LatentLds {
    static constexpr int K_ROW = KD * 32 + 8;                               // bf16 per key row
    static constexpr int BYTES = (AL_KEYS * K_ROW + DT * 16 * AL_VROW + DT * 2 * 32) * 2;
};

// A piece on its way from memory to LDS: a thread takes the two keys of a column (see above) and 8 numbers of both.
template <int KD, int DT>
struct LatentPiece {
    using L = LatentLds<KD, DT>;
    static constexpr int MAX_ITEMS = (AL_KEYS / 2) * (KD * 4) / 256 + 1;
    const bf16_t* cache; const int* pages; int dk, dv, tid;
    uint4 ra[MAX_ITEMS], rb[MAX_ITEMS];

    __device__ __forceinline__ void request(int piece) {
        const int key0 = piece * AL_KEYS, items = (AL_KEYS / 2) * (dk / 8);
        int phys = max(pages[key0 / AM_PAGE], 0);       // (a page that is not there holds no visible key)
        const bf16_t* base = cache + ((size_t)phys * AM_PAGE + key0 % AM_PAGE) * dk;
#pragma unroll
        for (int i = 0; i < MAX_ITEMS; ++i) {
            int w = tid + i * 256;
            if (w < items) {
                int c = w & 15, dc = w >> 4;            // 16 neighbouring lanes: the 16 columns, the same 8 numbers
                int ka = 8 * (c >> 2) + (c & 3);
                ra[i] = *(const uint4*)(base + (size_t)ka * dk + dc * 8);
                rb[i] = *(const uint4*)(base + (size_t)(ka + 4) * dk + dc * 8);
            }
        }
    }
    __device__ __forceinline__ void store(bf16_t* sk, bf16_t* sv) const {
        const int items = (AL_KEYS / 2) * (dk / 8), dv8 = dv / 8;
#pragma unroll
        for (int i = 0; i < MAX_ITEMS; ++i) {
            int w = tid + i * 256;
            if (w < items) {
                int c = w & 15, dc = w >> 4;
                *(uint4*)(sk + c * L::K_ROW + dc * 8) = ra[i];
                *(uint4*)(sk + (16 + c) * L::K_ROW + dc * 8) = rb[i];
                if (dc < dv8) {
                    const uint32_t a[4] = {ra[i].x, ra[i].y, ra[i].z, ra[i].w};
                    const uint32_t bw[4] = {rb[i].x, rb[i].y, rb[i].z, rb[i].w};
                    uint32_t* dst = (uint32_t*)(sv + al_vrow_at(dc * 8) + 2 * c);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        // numbers 2j and 2j + 1 of both keys, the two keys side by side
                        dst[(2 * j) * (AL_VROW / 2)] = (a[j] & 0xffffu) | (bw[j] << 16);
                        dst[(2 * j + 1) * (AL_VROW / 2)] = (a[j] >> 16) | (bw[j] & 0xffff0000u);
                    }
                }
            }
        }
    }
};

template <int KD, int DT, int RT>
__global__ void __launch_bounds__(256)
attn_latent_mfma_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
                        const int* __restrict__ block_table, int bt_width, const int* __restrict__ cu_seqlens,
                        int n_seqs, const int* __restrict__ token_pos, int n_heads, int dk, int dv,
                        float scale_log2e, int window, int n_splits, float* __restrict__ part_o,
                        float* __restrict__ part_ml) {
    using L = LatentLds<KD, DT>;
    extern __shared__ uint4 al_smem[];
    bf16_t* sk = (bf16_t*)al_smem;                    // [AL_KEYS][K_ROW]
    bf16_t* sv = sk + AL_KEYS * L::K_ROW;             // [DT * 16] rows at al_vrow_at
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int g = lane >> 4, col = lane & 15;
    int split = blockIdx.y;
    // which sequence and which of its row tiles
    int tile = blockIdx.x, b = 0, tok0 = 0, n_rows = 0;
    for (; b < n_seqs; ++b) {
        tok0 = cu_seqlens[b];
        n_rows = (cu_seqlens[b + 1] - tok0) * n_heads;
        int tiles = (n_rows + AL_ROWS * RT - 1) / (AL_ROWS * RT);
        if (tile < tiles) break;
        tile -= tiles;
    }
    if (b >= n_seqs) return;
    const int* pages = block_table + (size_t)b * bt_width;
    int pos0 = token_pos[tok0];
    int row0 = tile * AL_ROWS * RT, row1 = min(n_rows, row0 + AL_ROWS * RT) - 1;        // the block's rows
    int w_first = row0 + wave * 16 * RT, w_last = min(row1, w_first + 16 * RT - 1);    // the wave's rows
    bool wave_active = w_first <= row1;
    int wave_lo = window > 0 ? max(0, pos0 + w_first / n_heads - window + 1) : 0;     // first key any of the wave's rows sees
    int wave_hi = pos0 + w_last / n_heads;                                            // last key
    int blk_lo = window > 0 ? max(0, pos0 + row0 / n_heads - window + 1) : 0;
    int blk_hi = pos0 + row1 / n_heads;
    int first_piece = blk_lo / AL_KEYS, last_piece = blk_hi / AL_KEYS;

    // zeros where the sizes stop short of the tiles: they are never written again
    for (int i = tid; i < L::BYTES / 16; i += 256) al_smem[i] = make_uint4(0u, 0u, 0u, 0u);

    // Per tile of 16 rows: the lane's column is one row of work.  Q^T operand: 8 numbers per lane and step.
    bool row_ok[RT];
    int my_pos[RT], my_lo[RT];
    size_t grow[RT];
    bf16x8_t qf[RT][KD];
    float m[RT], l[RT];
    f32x4_t o[RT][DT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        int my_row = w_first + rt * 16 + col;
        row_ok[rt] = my_row <= row1;
        my_pos[rt] = pos0 + (row_ok[rt] ? my_row : row1) / n_heads;
        my_lo[rt] = window > 0 ? max(0, my_pos[rt] - window + 1) : 0;
        grow[rt] = (size_t)tok0 * n_heads + (row_ok[rt] ? my_row : row1);
        const bf16_t* qrow = q + grow[rt] * dk + g * 8;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) {
            bool ok = row_ok[rt] && kd * 32 + g * 8 < dk;
            uint4 v = ok ? *(const uint4*)(qrow + kd * 32) : make_uint4(0u, 0u, 0u, 0u);
            qf[rt][kd] = __builtin_bit_cast(bf16x8_t, v);
        }
        m[rt] = -INFINITY;
        l[rt] = 0.f;
#pragma unroll
        for (int i = 0; i < DT; ++i) o[rt][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    LatentPiece<KD, DT> next{cache, pages, dk, dv, tid};
    int piece = first_piece + split;
    if (piece <= last_piece) next.request(piece);
    for (; piece <= last_piece; piece += n_splits) {
        __syncthreads();                 // the piece before has been multiplied (first round: the zeros are written)
        next.store(sk, sv);
        __syncthreads();
        if (piece + n_splits <= last_piece) next.request(piece + n_splits);
        int key0 = piece * AL_KEYS;
        if (!wave_active || key0 > wave_hi || key0 + AL_KEYS - 1 < wave_lo) continue;      // wave-uniform
        // scores of 2 x 16 keys: row r of tile u is key 8 (r / 4) + 4 u + r % 4, so that element i of
        // s[rt][u] in lane (g, col) is key 8 g + 4 u + i of the column's row of work
        f32x4_t s[RT][2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) s[rt][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            const bf16_t* krow = sk + (16 * u + col) * L::K_ROW + g * 8;       // key 8 (col / 4) + 4 u + col % 4
#pragma unroll
            for (int kd = 0; kd < KD; ++kd) {
                bf16x8_t kf = __builtin_bit_cast(bf16x8_t, *(const uint4*)(krow + kd * 32));
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    s[rt][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[rt][kd], s[rt][u], 0, 0, 0);
            }
        }
        bf16x8_t pf[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float mx = -INFINITY;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int key = key0 + g * 8 + u * 4 + i;
                    float v = (row_ok[rt] && key >= my_lo[rt] && key <= my_pos[rt]) ? s[rt][u][i] * scale_log2e : -INFINITY;
                    s[rt][u][i] = v;
                    mx = fmaxf(mx, v);
                }
            mx = rows4_max(mx);
            // The exponents' reference m follows a row's maximum only when that has grown by more than
            // AL_LAZY_MAX: any reference gives the same quotient at the end, the probabilities stay below
            // 2^AL_LAZY_MAX, and the sums and outputs so far are rescaled only for a row's first pieces
            // instead of with every piece (the outputs are the bulk of a lane's registers).
            if (__builtin_amdgcn_ballot_w64(mx > m[rt] + AL_LAZY_MAX)) {
                float m_new = fmaxf(m[rt], mx);
                float corr = fast_exp2(m[rt] - (m_new == -INFINITY ? 0.f : m_new));
                l[rt] *= corr;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[rt][dt] = o[rt][dt] * corr;
                m[rt] = m_new;
            }
            float m_use = m[rt] == -INFINITY ? 0.f : m[rt];
            float sum = 0.f;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[rt][u][i] = fast_exp2(s[rt][u][i] - m_use);
                    sum += s[rt][u][i];
                }
            sum = rows4_sum(sum);
            l[rt] += sum;
            // P^T operand: slot 2 i + u = key 8 g + 4 u + i, the order of the transposed copy
            pf[rt] = __builtin_bit_cast(bf16x8_t, make_uint4(pack_bf16x2(s[rt][0][0], s[rt][1][0]), pack_bf16x2(s[rt][0][1], s[rt][1][1]),
                                                             pack_bf16x2(s[rt][0][2], s[rt][1][2]), pack_bf16x2(s[rt][0][3], s[rt][1][3])));
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            bf16x8_t vf = __builtin_bit_cast(bf16x8_t, *(const uint4*)(sv + al_vrow_at(dt * 16 + col) + g * 8));
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                o[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[rt], o[rt][dt], 0, 0, 0);
        }
    }
    // element i of o[rt][dt] is number 16 dt + 4 g + i of the column's row
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (!row_ok[rt]) continue;
        if (n_splits == 1) {
            float inv = 1.0f / l[rt];
            bf16_t* orow = out + grow[rt] * dv;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                int d = dt * 16 + 4 * g;
                if (d < dv)       // (dv is a multiple of 8: four numbers are inside or outside together)
                    *(uint2*)(orow + d) = make_uint2(pack_bf16x2(o[rt][dt][0] * inv, o[rt][dt][1] * inv),
                                                     pack_bf16x2(o[rt][dt][2] * inv, o[rt][dt][3] * inv));
            }
        } else {
            size_t slot = grow[rt] * n_splits + split;
            float* po = part_o + slot * dv;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                int d = dt * 16 + 4 * g;
                if (d < dv) *(float4*)(po + d) = make_float4(o[rt][dt][0], o[rt][dt][1], o[rt][dt][2], o[rt][dt][3]);
            }
            if (g == 0) {
                part_ml[slot * 2] = m[rt];
                part_ml[slot * 2 + 1] = l[rt];
            }
        }
    }
}

// A decode step whose sequences have at most 16 rows of work each: one block per sequence and split, whose four waves share the rows.  Of a piece's
// scores a wave forms 16 keys over half of the numbers, the halves meet in LDS, every wave forms the probabilities of all 32
// keys (the same in each) and a quarter of the output's numbers.  Bound by its chain of trips and barriers: with the rows in one
// wave (the other three only loading), the sequence looked up by one load after the other and the LDS zeroed ahead of every launch,
// 8 sequences of 2,048 keys (16 heads, 576 and 512 numbers) took 16.5 us, 13.3 this way (traced inside a step).  A split without a key writes no output: its weight is zero.
template <int KD, int DT>
__global__ void __launch_bounds__(256)
attn_latent_few_kernel(const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
                       const int* __restrict__ block_table, int bt_width, const int* __restrict__ cu_seqlens,
                       const int* __restrict__ token_pos, int n_heads, int dk, int dv,
                       float scale_log2e, int window, int n_splits, float* __restrict__ part_o,
                       float* __restrict__ part_ml) {
    using L = LatentLds<KD, DT>;
    constexpr int KH = (KD + 1) / 2, DW = DT / 4;     // steps of a half of the numbers, output tiles of a wave
    extern __shared__ uint4 al_smem[];
    __shared__ f32x4_t halves[2][2][64];              // [half of the numbers][16 keys]: sums of a wave
    bf16_t* sk = (bf16_t*)al_smem;
    bf16_t* sv = sk + AL_KEYS * L::K_ROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, col = lane & 15;
    const int b = blockIdx.x, split = blockIdx.y;
    const int tok0 = cu_seqlens[b], n_rows = (cu_seqlens[b + 1] - tok0) * n_heads, pos0 = token_pos[tok0];
    const int* pages = block_table + (size_t)b * bt_width;
    const bool row_ok = col < n_rows;
    const int my_pos = pos0 + min(col, n_rows - 1) / n_heads, my_lo = window > 0 ? max(0, my_pos - window + 1) : 0;
    const size_t grow = (size_t)tok0 * n_heads + min(col, n_rows - 1);
    const int lo = window > 0 ? max(0, pos0 - window + 1) : 0, hi = pos0 + (n_rows - 1) / n_heads;     // keys that any row sees
    const int last_piece = hi / AL_KEYS;
    int piece = lo / AL_KEYS + split;
    LatentPiece<KD, DT> next{cache, pages, dk, dv, tid};
    if (piece <= last_piece) next.request(piece);
    const int u_mine = wave & 1, half = wave >> 1;
    bf16x8_t qf[KH];
#pragma unroll
    for (int i = 0; i < KH; ++i) {
        const int at = (half * KH + i) * 32 + g * 8;
        uint4 v = row_ok && half * KH + i < KD && at < dk ? *(const uint4*)(q + grow * dk + at) : make_uint4(0u, 0u, 0u, 0u);
        qf[i] = __builtin_bit_cast(bf16x8_t, v);
    }
    if (dk < KD * 32 || dv < DT * 16) {               // zeros where the sizes stop short of the tiles: never written again
        for (int i = tid; i < L::BYTES / 16; i += 256) al_smem[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    float m = -INFINITY, l = 0.f;
    f32x4_t o[DW];
#pragma unroll
    for (int i = 0; i < DW; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const bool any = piece <= last_piece;
    for (; piece <= last_piece; piece += n_splits) {
        __syncthreads();                              // the piece before has been multiplied (first round: the zeros are written)
        next.store(sk, sv);
        __syncthreads();
        if (piece + n_splits <= last_piece) next.request(piece + n_splits);
        f32x4_t part = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const bf16_t* krow = sk + (16 * u_mine + col) * L::K_ROW + half * KH * 32 + g * 8;
#pragma unroll
        for (int i = 0; i < KH; ++i)
            if (half * KH + i < KD)
                part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, *(const uint4*)(krow + i * 32)), qf[i], part, 0, 0, 0);
        halves[half][u_mine][lane] = part;
        __syncthreads();
        f32x4_t s[2];
        float mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            s[u] = halves[0][u][lane] + halves[1][u][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = piece * AL_KEYS + g * 8 + u * 4 + i;
                s[u][i] = row_ok && key >= my_lo && key <= my_pos ? s[u][i] * scale_log2e : -INFINITY;
                mx = fmaxf(mx, s[u][i]);
            }
        }
        mx = rows4_max(mx);
        const float m_new = fmaxf(m, mx), m_use = m_new == -INFINITY ? 0.f : m_new, corr = fast_exp2(m - m_use);
        float sum = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[u][i] = fast_exp2(s[u][i] - m_use);
                sum += s[u][i];
            }
        sum = rows4_sum(sum);
        l = l * corr + sum;
        m = m_new;
        // P^T operand: slot 2 i + u = key 8 g + 4 u + i, the order of the transposed copy
        const bf16x8_t pf = __builtin_bit_cast(bf16x8_t, make_uint4(pack_bf16x2(s[0][0], s[1][0]), pack_bf16x2(s[0][1], s[1][1]),
                                                                     pack_bf16x2(s[0][2], s[1][2]), pack_bf16x2(s[0][3], s[1][3])));
#pragma unroll
        for (int i = 0; i < DW; ++i) {
            const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, *(const uint4*)(sv + al_vrow_at((wave * DW + i) * 16 + col) + g * 8));
            o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, o[i] * corr, 0, 0, 0);
        }
    }
    if (!row_ok) return;
    const size_t slot = grow * n_splits + split;
    if (n_splits > 1 && wave == 0 && g == 0) {
        part_ml[slot * 2] = m;
        part_ml[slot * 2 + 1] = l;
    }
    if (!any && n_splits > 1) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < DW; ++i) {
        const int d = (wave * DW + i) * 16 + 4 * g;   // (dv is a multiple of 8: four numbers are inside or outside together)
        if (d >= dv) continue;
        if (n_splits == 1) *(uint2*)(out + grow * dv + d) = make_uint2(pack_bf16x2(o[i][0] * inv, o[i][1] * inv), pack_bf16x2(o[i][2] * inv, o[i][3] * inv));
        else *(float4*)(part_o + slot * dv + d) = make_float4(o[i][0], o[i][1], o[i][2], o[i][3]);
    }
}

// Log-sum-exp merge of the splits of a row: one block per row.  At most 64 splits: lane s of every wave fetches split s's
// reference and sum, so these loads go out together.  GROUPS groups of threads, one for every eight splits, take every GROUPS th
// split each, four values a thread, all eight loads in one trip while the weights are formed, and meet in LDS in group order.
// A thread a value with the splits eight at a time was 14 trips at 51 splits of 512 values: 11.4 us, now 4.8.  Eight groups
// whatever the number of splits left most of a block idle where the rows are many and their splits few: 8,192 rows of 512
// values in two splits took 31 us longer.
template <int GROUPS>
__global__ void __launch_bounds__(128 * GROUPS)
attn_latent_reduce_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                          bf16_t* __restrict__ out, int n_splits, int dv) {
    extern __shared__ float alr_smem[];               // [64 weights][GROUPS][dv]
    float *wgt = alr_smem, *sums = alr_smem + 64;
    size_t row = blockIdx.x;
    const float* ml = part_ml + row * n_splits * 2;
    const float* po = part_o + row * n_splits * dv;
    const int lane = threadIdx.x & 63, quads = dv / 4;
    const int group = (int)threadIdx.x / quads, d = (int)threadIdx.x % quads * 4;   // (threads beyond the groups: group >= GROUPS)
    float2 mine = *(const float2*)(ml + 2 * min(lane, n_splits - 1));
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = *(const float4*)(po + (size_t)min(group + i * GROUPS, n_splits - 1) * dv + d);
    float ms = lane < n_splits ? mine.x : -INFINITY, ls = lane < n_splits ? mine.y : 0.f;
    float mm = wave_max(ms);
    float w = ms == -INFINITY ? 0.f : fast_exp2(ms - mm);
    if (threadIdx.x < 64) wgt[lane] = w;              // (zero beyond the last split)
    float inv_l = 1.0f / wave_sum(ls * w);            // every wave computes the same sum
    __syncthreads();
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    if (group < GROUPS) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int s = group + i * GROUPS;
            if (s >= n_splits) continue;
            float ws = wgt[s];
            if (ws == 0.f) continue;                  // (a split without a key has left nothing)
            acc.x = fmaf(v[i].x, ws, acc.x); acc.y = fmaf(v[i].y, ws, acc.y);
            acc.z = fmaf(v[i].z, ws, acc.z); acc.w = fmaf(v[i].w, ws, acc.w);
        }
        if (GROUPS > 1) *(float4*)(sums + group * dv + d) = acc;
    }
    if (GROUPS > 1) {
        __syncthreads();
        if (group == 0) {
#pragma unroll
            for (int g = 1; g < GROUPS; ++g) {
                float4 u = *(const float4*)(sums + g * dv + d);
                acc.x += u.x; acc.y += u.y; acc.z += u.z; acc.w += u.w;
            }
        }
    }
    if (group != 0) return;
    *(uint2*)(out + row * dv + d) = make_uint2(f32x2_to_bf16x2(acc.x * inv_l, acc.y * inv_l), f32x2_to_bf16x2(acc.z * inv_l, acc.w * inv_l));
}

template <int GROUPS>
static void launch_latent_reduce(const float* part_o, const float* part_ml, bf16_t* out, long long rows, int n_splits, int dv, hipStream_t stream) {
    attn_latent_reduce_kernel<GROUPS><<<(unsigned)rows, (GROUPS * (dv / 4) + 63) / 64 * 64, (64 + (GROUPS > 1 ? GROUPS * dv : 0)) * sizeof(float), stream>>>(
        part_o, part_ml, out, n_splits, dv);
}
