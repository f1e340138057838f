// Attention over the paged 32-bit cache on the 32-bit matrix instructions (v_mfma_f32_16x16x4_f32: full 32-bit products and
// sums).  The plain kernel (attention_generic.h), a row of keys per thread, takes 36 ms of attention in a pass of 574 prompt
// tokens and 15 decode steps of four sequences through 28 layers of Qwen3-0.6B (16 heads of 128); these take 8.3.
//
// A wave works on 16 rows, a row being a (token, query head) of one key/value head; keys come a page of 64 at a time.
// S^T = K Q^T: lane l holds the scores of row l%16 with the keys 16 t + 4 (l/16) + e of the page.  That is the layout in
// which the next product O^T = V^T P^T takes its probabilities, so they go from one to the other in registers; a lane reads
// four neighbouring numbers of a key or value row at once and multiplies them one after the other, the same places of both
// operands each time.  The running maximum, sum and output of a row live in the four lanes l%16 + 16 g.
//  * attn_f32_prompt_kernel: 64 rows a block, a wave 16 of them; keys and values of a page pass through LDS.  Bound by the
//    matrix cores (8,192 clocks a page and SIMD at head size 128 against 2,048 of the LDS).
//  * attn_f32_token_kernel: the heads of one token (up to 16 rows), the block's waves share out the keys in tiles of 16 and read
//    them straight from memory; they meet in LDS at the end, in wave order.  Bound by trips to memory: whole pages a wave
//    took 28 us at 315 keys, tiles of 16, whose
//    keys and values come in one trip, take 16.8.
// Masks as in attention_generic.h: window with kept first positions, or blocks of positions; slopes, sinks, soft cap.
#pragma once
#include "attention_generic.h"

typedef __attribute__((ext_vector_type(4))) float af_f32x4_t;
constexpr int AF_PAGE = 64;

struct AttnF32Args {
    const float *q, *kcache, *vcache;
    float* out;
    const int *block_table, *token_seq, *token_pos, *cu_seqlens;
    int bt_width, hq, hkv, window;
    float scale;
    AttnExtra ex;
    int few = 0;                // with both kernels: sequences of at most so many query tokens are the token kernel's
};

// Scores of 16 rows with NT tiles of 16 keys: krow(t, c) is the lane's piece (16 c + 4 (l/16) .. + 3) of key 16 t + l%16,
// query(c) that of its row.
template <int KD, int NT, typename Query, typename Row>
__device__ __forceinline__ void af_scores(Query query, Row krow, af_f32x4_t (&s)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        // two sums, of the even and the odd places: a product waits 32 clocks for the one before it in its sum
        af_f32x4_t odd = {0.f, 0.f, 0.f, 0.f};
        s[t] = odd;
#pragma unroll
        for (int c = 0; c < KD; ++c) {
            af_f32x4_t a = krow(t, c), q = query(c);
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], q[e], s[t], 0, 0, 0);
                odd = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e + 1], q[e + 1], odd, 0, 0, 0);
            }
        }
        s[t] += odd;
    }
}

// Masks the scores, moves the row's maximum and turns the scores into probabilities.  l is this lane's share of the sum.
template <int KD, int NT>
__device__ __forceinline__ void af_softmax(af_f32x4_t (&s)[NT], af_f32x4_t (&o)[KD], float& m, float& l, const AttnF32Args& a,
                                           int first_key, int lane, int pos, int lo, float slope) {
    float top = -INFINITY;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int key = first_key + t * 16 + (lane >> 4) * 4 + e;
            float v = s[t][e] * a.scale;
            if (a.ex.softcap > 0.f) v = a.ex.softcap * tanhf(v / a.ex.softcap);
            v -= slope * (float)(pos - key);
            bool seen = key <= pos && (key >= lo || key < a.ex.keep_first);
            s[t][e] = seen ? v : -INFINITY;
            top = fmaxf(top, s[t][e]);
        }
    top = rows4_max(top);
    float m_new = fmaxf(m, top);
    float ref = m_new == -INFINITY ? 0.f : m_new;     // nothing seen yet: every probability is exp(-inf)
    float corr = expf(m - ref);
    l *= corr;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[t][e] = expf(s[t][e] - ref);
            l += s[t][e];
        }
#pragma unroll
    for (int c = 0; c < KD; ++c) o[c] *= corr;
    m = m_new;
}

// o[c][e]: value 16 c + 4 (l/16) + e of row l%16; vrow(c, t) is the lane's piece of value row 16 c + l%16 at the keys
// 16 t + 4 (l/16) .. + 3.
template <int KD, int NT, typename Row>
__device__ __forceinline__ void af_values(const af_f32x4_t (&p)[NT], Row vrow, af_f32x4_t (&o)[KD]) {
#pragma unroll
    for (int c = 0; c < KD; ++c)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            af_f32x4_t a = vrow(c, t);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], p[t][e], o[c], 0, 0, 0);
        }
}

__device__ __forceinline__ bool af_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// Adds what the page's infinite and NaN values give the rows that see their keys; every other value has had its product.
// values: the page's [D][64] in memory.
template <int KD>
__device__ __forceinline__ void af_add_odd_values(const af_f32x4_t (&p)[4], const float* values, af_f32x4_t (&o)[KD], const AttnF32Args& a,
                                                  int first_key, int lane, int pos, int lo) {
#pragma unroll 1
    for (int k = 0; k < AF_PAGE; ++k) {
        float mine = 0.f;                             // the probability that lane l%16 + 16 (k%16 / 4) holds of key k
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine = t * 16 + e == (k & ~12) ? p[t][e] : mine;
        const float w = __shfl(mine, (lane & 15) + (k & 12) * 4, 64);
        const int key = first_key + k;
        const bool seen = key <= pos && (key >= lo || key < a.ex.keep_first);
        int at = (lane >> 4) * 4 * AF_PAGE + k;
        asm volatile("" : "+v"(at));                  // (addresses formed before the loop, or all loads at once, would take
#pragma unroll                                        //  registers that the kernel is short of)
        for (int c = 0; c < KD; ++c) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = values[at + (c * 16 + e) * AF_PAGE];
                if (seen && !af_finite(v)) o[c][e] = fmaf(w, v, o[c][e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// (registers for as many blocks as find room in a CU's LDS)
constexpr int af_prompt_lds(int d) { return (AF_PAGE * (d + 4) + d * (AF_PAGE + 4) + 4) * 4; }
constexpr int af_prompt_blocks(int d) { return 160 * 1024 / af_prompt_lds(d) < 4 ? 160 * 1024 / af_prompt_lds(d) : 4; }

template <int KD>
__global__ void __launch_bounds__(256, af_prompt_blocks(KD * 16))
attn_f32_prompt_kernel(AttnF32Args a) {
    constexpr int D = KD * 16, KS = D + 4, VS = AF_PAGE + 4;      // padded rows: 16 rows fall into different banks
    extern __shared__ float af_smem[];
    float *ks = af_smem, *vs = af_smem + AF_PAGE * KS;
    float& odd_page = vs[D * VS];                     // the last page that holds an infinite or NaN value (a variable of its own
                                                      // before the rows would put them at an odd multiple of 4 bytes, and one
                                                      // that is no float would make the page table's reads vector loads)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int seq = blockIdx.y, kvh = blockIdx.z, group = a.hq / a.hkv;
    const int t0 = a.cu_seqlens[seq], count = a.cu_seqlens[seq + 1] - t0;
    const int row0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * 64, n_rows = count * group;   // the longest rows first
    if (row0 >= n_rows || count <= a.few) return;
    const int row = min(row0 + wave * 16 + (lane & 15), n_rows - 1);
    const int t = t0 + row / group, h = kvh * group + row % group;
    const int pos = a.token_pos[t], lo = attn_first_key(pos, a.window, a.ex.chunk);
    const int last_pos = a.token_pos[t0 + min(row0 + 63, n_rows - 1) / group];
    const int lo_page = attn_first_key(a.token_pos[t0 + row0 / group], a.window, a.ex.chunk) / AF_PAGE;
    const int kept_pages = (a.ex.keep_first + AF_PAGE - 1) / AF_PAGE;
    const int* pages = a.block_table + (size_t)seq * a.bt_width;
    const float slope = a.ex.slopes ? a.ex.slopes[h] : 0.f;
    af_f32x4_t q[KD], o[KD], s[4];
#pragma unroll
    for (int c = 0; c < KD; ++c) {
        q[c] = *(const af_f32x4_t*)(a.q + ((size_t)t * a.hq + h) * D + c * 16 + (lane >> 4) * 4);
        o[c] = af_f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    float m = -INFINITY, l = 0.f;
    if (threadIdx.x == 0) odd_page = -1.f;
    for (int p = 0; p <= last_pos / AF_PAGE; ++p) {
        if (p >= kept_pages && p < lo_page) continue;
        const size_t at = ((size_t)pages[p] * a.hkv + kvh) * AF_PAGE * D;
        // Values behind `known` are another sequence's, if any.  The page's values meet the probabilities of 16 rows at once,
        // and zero times infinity is NaN: a row must not see the infinite or NaN value of a key it does not see (a later
        // token's, or one before its window).  Such values are taken out of the page and added to the rows that see them.
        const int known = last_pos - p * AF_PAGE;
        __syncthreads();
        float odd = 0.f;                              // NaN once a value was infinite or NaN
        for (int i = threadIdx.x; i < AF_PAGE * D / 4; i += 256) {
            *(af_f32x4_t*)(ks + i / (D / 4) * KS + i % (D / 4) * 4) = *(const af_f32x4_t*)(a.kcache + at + i * 4);
            af_f32x4_t v = *(const af_f32x4_t*)(a.vcache + at + i * 4);
            int key = i % (AF_PAGE / 4) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = key + e <= known ? v[e] : 0.f;
                odd = fmaf(v[e], 0.f, odd);
            }
            *(af_f32x4_t*)(vs + i / (AF_PAGE / 4) * VS + key) = v;
        }
        if (!(odd == 0.f)) odd_page = (float)p;
        __syncthreads();
        const bool repair = odd_page == (float)p;
        if (repair) {
            for (int i = threadIdx.x; i < AF_PAGE * D; i += 256) {
                float& v = vs[i / AF_PAGE * VS + i % AF_PAGE];
                if (!af_finite(v)) v = 0.f;
            }
            __syncthreads();
        }
        af_scores<KD, 4>([&](int c) { return q[c]; }, [&](int kt, int c) { return *(const af_f32x4_t*)(ks + (kt * 16 + (lane & 15)) * KS + c * 16 + (lane >> 4) * 4); }, s);
        af_softmax<KD, 4>(s, o, m, l, a, p * AF_PAGE, lane, pos, lo, slope);
        af_values<KD, 4>(s, [&](int c, int kt) { return *(const af_f32x4_t*)(vs + (c * 16 + (lane & 15)) * VS + kt * 16 + (lane >> 4) * 4); }, o);
        if (repair) af_add_odd_values<KD>(s, a.vcache + at, o, a, p * AF_PAGE, lane, pos, lo);
    }
    l = rows4_sum(l);
    float down = 1.f;
    if (a.ex.sink) {
        float sink = a.ex.sinks ? a.ex.sinks[h] : 0.f, top = fmaxf(m, sink);
        down = expf(m - top);
        l = l * down + expf(sink - top);
    }
    if (row0 + wave * 16 + (lane & 15) >= n_rows) return;
    float* to = a.out + ((size_t)t * a.hq + h) * D + (lane >> 4) * 4;
#pragma unroll
    for (int c = 0; c < KD; ++c) {
        af_f32x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = o[c][e] * down / l;
        *(af_f32x4_t*)(to + c * 16) = v;
    }
}

template <int KD, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
attn_f32_token_kernel(AttnF32Args a) {
    constexpr int D = KD * 16, ROW = D + 4;
    extern __shared__ float af_smem[];                // [WAVES][16][ROW], then maxima and sums [WAVES][16] each, then [16][ROW] queries
    float *os = af_smem, *ms = af_smem + WAVES * 16 * ROW, *ls = ms + WAVES * 16, *qs = ls + WAVES * 16;
    // Sixteen waves leave 128 registers a lane, which keys, values, queries and sums of 128 numbers a head fill: the queries
    // stay in LDS then (in registers, seven others were spilled; 64 sequences of 1,000 keys: 118 and 105 us).
    constexpr bool Q_IN_LDS = WAVES == 16 && KD == 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kvh = blockIdx.y, group = a.hq / a.hkv, g0 = blockIdx.z * 16;
    int t = blockIdx.x;
    if (a.few) {                                      // blocks for `few` tokens of every sequence
        const int seq = t / a.few, at = t % a.few, t0 = a.cu_seqlens[seq], count = a.cu_seqlens[seq + 1] - t0;
        if (count > a.few || at >= count) return;
        t = __builtin_amdgcn_readfirstlane(t0 + at);
    }
    const int h = kvh * group + min(g0 + (lane & 15), group - 1);
    const int pos = a.token_pos[t], lo = attn_first_key(pos, a.window, a.ex.chunk);
    const int* pages = a.block_table + (size_t)a.token_seq[t] * a.bt_width;
    const float slope = a.ex.slopes ? a.ex.slopes[h] : 0.f;
    af_f32x4_t q[KD], o[KD], s[1];
#pragma unroll
    for (int c = 0; c < KD; ++c) {
        if (!Q_IN_LDS) q[c] = *(const af_f32x4_t*)(a.q + ((size_t)t * a.hq + h) * D + c * 16 + (lane >> 4) * 4);
        o[c] = af_f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    if (Q_IN_LDS) {
        for (int c = wave; c < KD; c += WAVES)
            *(af_f32x4_t*)(qs + (lane & 15) * ROW + c * 16 + (lane >> 4) * 4) =
                *(const af_f32x4_t*)(a.q + ((size_t)t * a.hq + h) * D + c * 16 + (lane >> 4) * 4);
        __syncthreads();
    }
    float m = -INFINITY, l = 0.f;
    // the pages of the kept first positions, then those of the window
    const int last_page = pos / AF_PAGE, lo_page = lo / AF_PAGE;
    const int kept_pages = min((a.ex.keep_first + AF_PAGE - 1) / AF_PAGE, lo_page);
    const int n_tiles = (kept_pages + last_page - lo_page + 1) * (AF_PAGE / 16);
    for (int i = wave; i < n_tiles; i += WAVES) {
        const int listed = i / (AF_PAGE / 16), in_page = i % (AF_PAGE / 16) * 16;
        const int p = listed < kept_pages ? listed : lo_page + listed - kept_pages, first = p * AF_PAGE + in_page;
        if (first > pos || (first + 15 < lo && first >= a.ex.keep_first)) continue;
        const size_t at = ((size_t)pages[p] * a.hkv + kvh) * AF_PAGE * D;
        const float *kp = a.kcache + at + (size_t)(in_page + (lane & 15)) * D + (lane >> 4) * 4;
        const float *vp = a.vcache + at + (size_t)(lane & 15) * AF_PAGE + in_page + (lane >> 4) * 4;
        // keys and values are asked for together: one trip to memory a tile
        af_f32x4_t k[KD], v[KD];
#pragma unroll
        for (int c = 0; c < KD; ++c) k[c] = *(const af_f32x4_t*)(kp + c * 16);
        if (KD <= 8)
#pragma unroll
            for (int c = 0; c < KD; ++c) v[c] = *(const af_f32x4_t*)(vp + c * 16 * AF_PAGE);
        if constexpr (Q_IN_LDS)
            af_scores<KD, 1>([&](int c) { return *(const af_f32x4_t*)(qs + (lane & 15) * ROW + c * 16 + (lane >> 4) * 4); },
                             [&](int, int c) { return k[c]; }, s);
        else
            af_scores<KD, 1>([&](int c) { return q[c]; }, [&](int, int c) { return k[c]; }, s);
        if (KD > 8)                                   // (beyond 128 numbers a head both do not fit the registers)
#pragma unroll
            for (int c = 0; c < KD; ++c) v[c] = *(const af_f32x4_t*)(vp + c * 16 * AF_PAGE);
        af_softmax<KD, 1>(s, o, m, l, a, first, lane, pos, lo, slope);
        bool seen[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int key = first + (lane >> 4) * 4 + e;
            seen[e] = key <= pos && (key >= lo || key < a.ex.keep_first);
        }
        af_values<KD, 1>(s, [&](int c, int) {
            af_f32x4_t u = v[c];                      // a key that is not seen may hold anything: it is left out, not weighted by zero
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] = seen[e] ? u[e] : 0.f;
            return u;
        }, o);
    }
    l = rows4_sum(l);
    if (lane < 16) {
        ms[wave * 16 + lane] = m;
        ls[wave * 16 + lane] = l;
    }
#pragma unroll
    for (int c = 0; c < KD; ++c) *(af_f32x4_t*)(os + (wave * 16 + (lane & 15)) * ROW + c * 16 + (lane >> 4) * 4) = o[c];
    __syncthreads();
    const int rows = min(group - g0, 16);
    for (int i = threadIdx.x; i < rows * (D / 4); i += 64 * WAVES) {
        const int r = i / (D / 4), e = i % (D / 4) * 4, head = kvh * group + g0 + r;
        float top = -INFINITY;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) top = fmaxf(top, ms[w * 16 + r]);
        float sum = 0.f;
        if (a.ex.sink) {
            float sink = a.ex.sinks ? a.ex.sinks[head] : 0.f;
            top = fmaxf(top, sink);
            sum = expf(sink - top);
        }
        af_f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            float f = expf(ms[w * 16 + r] - top);     // a wave without a page: exp(-inf)
            sum += ls[w * 16 + r] * f;
            v += *(const af_f32x4_t*)(os + (w * 16 + r) * ROW + e) * f;
        }
        *(af_f32x4_t*)(a.out + ((size_t)t * a.hq + head) * D + e) = v / sum;
    }
}

// Microseconds of both kernels over a step whose sequences have counts[b] query tokens (each `all` without counts) when those
// of at most `few` go to the token kernel.  A page costs a block of 64 rows about 1 us per 16 numbers of a head and a block of
// one token a quarter of it (its waves share the page), half as much again where the blocks are more than the CUs; measured
// at heads of 32, 128 and 256: 1.4, 1.0 and 0.9, and 0.27 at all three.  How far back a sequence reaches is known of the longest
// one only (`pages`): up to 64 tokens are taken to stand at the end of so much, more of them to be a whole prompt.
static double af_cost(int few, const int* counts, int n_seqs, int all, int pages, int d, int group, int hkv, int cus) {
    struct { double work = 0.0, longest = 0.0; } rows, token;       // pages of all blocks, and of the longest
    for (int b = 0; b < n_seqs; ++b) {
        int c = counts ? counts[b] : all;
        if (c == 0) continue;
        double reach = n_seqs == 1 || c <= AF_PAGE || ceil_div(c, AF_PAGE) > pages ? pages : ceil_div(c, AF_PAGE);
        auto& k = c <= few ? token : rows;
        k.work += reach * hkv * (c <= few ? (double)c * ceil_div(group, 16) : (double)ceil_div((long long)c * group, 64));
        if (reach > k.longest) k.longest = reach;
    }
    double t = 0.0, page = d / 16.0;
    if (rows.work > 0.0) t += 6.0 + page * (rows.work > cus * rows.longest ? rows.work / cus : rows.longest);
    if (token.work > 0.0) t += 6.0 + 0.25 * page * (token.work > cus * token.longest ? 1.5 * token.work / cus : token.longest);
    return t;
}

// The line between the two kernels for a step: the cheapest of the powers of two, none and all.  Blocks of 64 rows pay for
// prompts; a few tokens behind a long context, or one token a sequence beside a prompt, leave them nearly empty and few, each
// walking all pages by itself.  Microseconds at 8 heads of 256 on 2: 5 tokens behind 1,000 positions 196 in blocks of 64 rows,
// 64 by token; 5 new ones 18 and 8; 300 ones beside 15 sequences of one token and 2,000 positions 481, and 232 with both kernels.
static int af_few(const AttnF32Args& a, int d, const int* counts, int n_seqs, int max_new, int max_len, int cus) {
    const int group = a.hq / a.hkv;
    int pages = max_len > 0 ? ceil_div(max_len, AF_PAGE) : a.bt_width;
    const int span = a.window > 0 ? a.window : a.ex.chunk;
    if (span > 0) {
        int seen = ceil_div(span, AF_PAGE) + 1 + ceil_div(a.ex.keep_first, AF_PAGE);
        if (seen < pages) pages = seen;
    }
    int best = max_new;
    double best_t = af_cost(max_new, counts, n_seqs, max_new, pages, d, group, a.hkv, cus);
    for (long long few = 0; few < max_new && few <= 4096; few = few ? 2 * few : 1) {
        double t = af_cost((int)few, counts, n_seqs, max_new, pages, d, group, a.hkv, cus);
        if (t < best_t) { best = (int)few; best_t = t; }
    }
    return best;
}

template <int KD>
static int launch_attn_f32(AttnF32Args a, int n_tokens, const int* counts, int n_seqs, int max_new, int max_len, int cus, hipStream_t stream) {
    constexpr int D = KD * 16;
    const int group = a.hq / a.hkv;
    constexpr int PROMPT_LDS = af_prompt_lds(D);
    constexpr int MANY = D <= 128 ? 16 : 8;           // (registers: a tile's keys and values, the queries and the sums)
    constexpr int FEW_LDS = 4 * 16 * (D + 6) * 4, MANY_LDS = MANY * 16 * (D + 6) * 4 + (MANY == 16 && D == 128 ? 16 * (D + 4) * 4 : 0);
    static bool ready = false;
    if (!ready) {
        const struct { const void* f; int bytes; } all[] = {{(const void*)attn_f32_prompt_kernel<KD>, PROMPT_LDS},
                                                            {(const void*)attn_f32_token_kernel<KD, 4>, FEW_LDS},
                                                            {(const void*)attn_f32_token_kernel<KD, MANY>, MANY_LDS}};
        for (const auto& k : all)
            if (hipFuncSetAttribute(k.f, hipFuncAttributeMaxDynamicSharedMemorySize, k.bytes) != hipSuccess)
                return rocml_fail("attention: cannot reserve %d bytes of LDS", k.bytes);
        ready = true;
    }
    const int few = a.cu_seqlens && n_seqs > 0 && max_new > 1 ? af_few(a, D, counts, n_seqs, max_new, max_len, cus) : 0x7fffffff;
    long long by_token = 0, by_rows = 0;              // tokens of either kernel
    for (int b = 0; few < max_new && b < n_seqs; ++b) {
        int c = counts ? counts[b] : max_new;
        (c <= few ? by_token : by_rows) += c;
    }
    // (a kernel that runs alone takes every sequence, whatever its count: a recorded step may be replayed with others)
    if (by_rows > 0) {
        if (by_token > 0) a.few = few;
        dim3 grid(ceil_div((long long)max_new * group, 64), n_seqs, a.hkv);
        attn_f32_prompt_kernel<KD><<<grid, 256, PROMPT_LDS, stream>>>(a);
        if (by_token == 0) return 0;
    } else {
        by_token = n_tokens;
    }
    // Waves a block by the room of the block table, which a recorded step keeps as its sequences grow: more than four where
    // the pages are many and the blocks are not.
    dim3 grid(a.few ? n_seqs * a.few : n_tokens, a.hkv, ceil_div(group, 16));
    if (a.bt_width >= 8 && by_token * a.hkv <= 2ll * cus)
        attn_f32_token_kernel<KD, MANY><<<grid, 64 * MANY, MANY_LDS, stream>>>(a);
    else
        attn_f32_token_kernel<KD, 4><<<grid, 256, FEW_LDS, stream>>>(a);
    return 0;
}
