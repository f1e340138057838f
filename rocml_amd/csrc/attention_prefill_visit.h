// A visit of a page by a block of attn_prefill_mfma_kernel, whose names it uses: into LDS, scores, softmax, values.  AM_LEAVE leaves it.
const int lpage = logical_page(visit);
__syncthreads();                                // the previous page has been consumed
#pragma unroll
for (int i = 0; i < K_PIECES; ++i) {
    int piece = tid + i * AM_THREADS;
    int key = piece / (D / 8), dc = piece % (D / 8);
    *(u32x4*)(sk + key * L::K_ROW + dc * 8) = kreg[i];
}
#pragma unroll
for (int i = 0; i < V_PIECES; ++i) {
    int piece = tid + i * AM_THREADS;
    // Within 16 keys the four groups of 4 stand in the order 0, 2, 1, 3: the second product
    // wants keys {4h .. 4h+3, 8+4h .. 8+4h+3} per lane (the order the scores come in), and
    // so finds them side by side, one 16-byte read.
    int d = piece / 8, kc = piece % 8;
    uint2* dst = (uint2*)(sv + d * L::V_ROW + (kc >> 1) * 16 + (kc & 1) * 4);
    dst[0] = make_uint2(vreg[i][0], vreg[i][1]);
    dst[2] = make_uint2(vreg[i][2], vreg[i][3]);
}
__syncthreads();
if (visit + 1 < n_visits) AM_LOAD_PAGE(logical_page(visit + 1))
if (!wave_active) AM_LEAVE;
// The scores of both 32-key halves are started before either is finished: the softmax of
// the first half (vector ALU) then runs while the matrix core still multiplies the second,
// and the softmax of the second while the first half's values are multiplied.
// S^T: element e of s is key 8(e/4) + 4 h2 + e%4, column = query row.
int page_key0 = lpage * AM_PAGE;
bool live[2];
f32x16_t sc[2];
#pragma unroll
for (int half = 0; half < 2; ++half) {
    int key0 = page_key0 + half * 32;
    live[half] = !(key0 > wave_last_key || (key0 + 31 < wave_first_key && !(EXTRA && key0 < keep)));   // wave-uniform
    if (!live[half]) continue;
#pragma unroll
    for (int e = 0; e < 16; ++e) sc[half][e] = 0.f;
    const bf16_t* krow = sk + (half * 32 + col) * L::K_ROW + h2 * 8;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
        bf16x8_t kf = __builtin_bit_cast(bf16x8_t, *(const uint4*)(krow + kk * 16));
        sc[half] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[kk], sc[half], 0, 0, 0);
    }
}
__builtin_amdgcn_sched_barrier(0);
#pragma unroll
for (int half = 0; half < 2; ++half) {
    if (!live[half]) continue;
    int key0 = page_key0 + half * 32;
    f32x16_t& s = sc[half];
    bool need_mask = !wave_full || key0 + 31 > wave_min_pos || key0 < wave_max_lo;   // wave-uniform
    if constexpr (EXTRA) {
        if (cap_out != 0.f) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = am_tanh(s[e] * cap_in) * cap_out;
        }
    }
    if (need_mask) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            int key = key0 + 8 * (e >> 2) + 4 * h2 + (e & 3);
            s[e] = (row_ok && key <= my_pos && (key >= my_lo || (EXTRA && key < keep))) ? s[e] : -INFINITY;
        }
    }
    if constexpr (EXTRA) {
        if (kslope != 0.f) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                int key = key0 + 8 * (e >> 2) + 4 * h2 + (e & 3);
                s[e] -= kslope * (float)(my_pos - key);
            }
        }
    }
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    mx = max_across_halves(mx) * scale_log2e;       // the scale is positive
    // The exponents' reference m follows a row's maximum only when that has grown by more
    // than AM_LAZY_MAX (powers of two): any reference gives the same quotient at the end,
    // the probabilities stay below 2^AM_LAZY_MAX, which bfloat16 and the 32-bit sums hold
    // with room to spare, and the sums and outputs so far have to be rescaled (64 products
    // a lane) only for the first pieces of a row instead of whenever one of a wave's 32
    // rows meets a new maximum, which with a thousand keys behind it is still every other piece.
    if (__builtin_amdgcn_ballot_w64(mx > m + AM_LAZY_MAX)) {
        float m_new = fmaxf(m, mx);
        float corr = fast_exp2(m - (m_new == -INFINITY ? 0.f : m_new));
        l *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] *= corr;
        m = m_new;
    }
    float m_use = m == -INFINITY ? 0.f : m;
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        s[e] = fast_exp2(fmaf(s[e], scale_log2e, -m_use));
        sum += s[e];
    }
    sum = sum_across_halves(sum);
    l += sum;
    // P^T operands: MFMA u takes elements 8u..8u+7 = keys 16u + {4 h2 .. +3, 8 + 4 h2 .. +3}.
    bf16x8_t pf[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
        pf[u] = __builtin_bit_cast(bf16x8_t, make_uint4(
            pack_bf16x2(s[8 * u + 0], s[8 * u + 1]), pack_bf16x2(s[8 * u + 2], s[8 * u + 3]),
            pack_bf16x2(s[8 * u + 4], s[8 * u + 5]), pack_bf16x2(s[8 * u + 6], s[8 * u + 7])));
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const bf16_t* vrow = sv + (dt * 32 + col) * L::V_ROW + half * 32 + 16 * u + 8 * h2;
            bf16x8_t vf = __builtin_bit_cast(bf16x8_t, *(const uint4*)vrow);
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[u], o[dt], 0, 0, 0);
        }
    }
}
