// A decode step's layers in one launch (gfx950, wave64, bfloat16 and 32-bit): q/k/v projection, attention over the paged cache,
// output projection, gated feed-forward, layer after layer, for one to four sequences of a model with small layers.
//
// What bounds it, and why it is one launch.  With a few rows of activations every product is a walk over its weights, and a
// step used to be five or six dependent kernels a layer.  A kernel that follows another starts with nothing on its way to it:
// launch, the first trip to memory and the last store are 4 to 5 us beside its bytes, and the weights, which depend on nothing,
// wait with everything else.  Here a block (one a CU) takes the products' tiles and the attentions' heads of all layers in the
// order in which they depend on each other: it asks for its weights (or its pages) first, then waits for its operands, so that
// the next stages' weights are in registers while this stage's results travel.  From a block's store to the waiting blocks that
// read it some 1.5 us pass.  A step of the Qwen3-0.6B shape (28 layers, replayed, to the logits): one sequence of 40 tokens
// 869 -> 437 us, of 500 938 -> 485, of 5,000 1,024 -> 749; two of 2,000 1,003 -> 650; four of 300 976 -> 660 (with how many keys it is
// slower: rocml_decode_chain_reach).  What is left of a layer (some 13 us) is five times a result's way to the next stage (1 to 1.5 us from its
// store to the operands behind it), 0.6 to 1 us of products and 0.3 to 0.6 of an epilogue.
//
// Measured on the way: two and three blocks a CU instead of one, 657 and 678 us against 558 (more weights ahead, but what asks
// for operands is in the way of what answers); eight waves a block 648 against 548 (but see dc_plan); a wave of its own for
// operands and results 994; a counter of flags beside plain data instead of words that carry their number 4.2 us from stage to
// stage against 2.1; one counter of tickets for all 30 ns a ticket, 24 us a layer.
//
// Operands travel between blocks as 64-bit words {32 bits of data, 32 bits of the launch's and layer's number}, written and
// read as relaxed atomics of agent scope, which pass by the L2s that the eight dies do not share: a word is either there whole
// or not yet, so no flag, fence or order between words is needed.  A buffer is written again a layer later at the earliest:
// its readers have then all published something that the writer's operands came from.  (Numbers repeat after 2^27 launches.)
//
// No wait can last: an item's place in the order is a ticket that a running block draws, and it waits only for items with lower
// tickets.  The items are dealt over eight counters; of each counter's tickets the lowest unfinished one is held by a block that
// runs and waits for nothing but finished items, or is the next that a running block draws.  That needs one running block for
// each counter: a block gets its counter when it starts, in turn, so any eight running blocks of a launch are enough, whatever
// else the GPU runs.  (By its place in the grid, which saves up to 1 % of a step, it would not do: a die starts its eighth of a grid by
// itself, and of two such launches side by side each could fill a die that the other's blocks of one counter wait for.)  Should a
// wait last for seconds all the same, it ends, and the step's result is NaN: it leaves the launch's number as a mark, so that the
// launch's other waits end too, while the next launch waits as if nothing had been, and tells the host (late).
//
// The algebra is that of the kernels the step otherwise runs (gemm_kpar_kernel, gemm_residual_prescale_kernel,
// attn_decode_mfma_kernel FUSED; gemm_f32_rows_kernel, attn_f32_token_kernel): 32-bit sums, the residual stream in 32 bits, the
// norm's scale applied by the consumer of bfloat16(x * gain), partial results of key splits merged in split order.
//
// A library of its own: a model that has no such layers does not load these kernels with those of its attention.
#include "common.h"
#include "attention_generic.h"
#include "attention_f32.h"
#include "attention_mfma.h"

ROCML_LAST_ERROR_FN(decode_chain)

typedef unsigned long long u64;
typedef __attribute__((ext_vector_type(4))) uint32_t dc_u32x4_t;

constexpr int DC_LAYERS = 32;           // layers of a launch (their pointers are kernel arguments)
constexpr int DC_MAX_ROWS = 4;
constexpr int DC_SHARDS = 8, DC_LINE = 16;      // ticket counters, 64-bit words between two of them (a line)
constexpr int DC_D = 128;               // head size
constexpr int DC_MAX_GROUP = 8;
constexpr int DC_GROUP = 4;             // loads of 16 bytes a lane asked for together
constexpr int DC_RING = 6;              // such groups on their way
constexpr int DC_TILE = 16;             // weight rows of a tile
constexpr int DC_MAX_TILES = 3;         // tiles of a block whose K is short
constexpr int DC_MAX_LDS = 128 << 10;
// words between two tiles' sums of squares (side by side, sixteen blocks write one line that all ask for: 24 against 20 us a layer)
constexpr int DC_APART = 8;
constexpr int DC_PAD = 64;              // bytes between two rows of activations in LDS
constexpr long long DC_PATIENCE = 400000000ll;  // ticks of 10 ns after which a wait gives up
constexpr int DC_POLLS = 256;                   // looks at a word between two looks at the clock and the mark (a power of two)

// The compute type's ways.  bfloat16: two values a word of operands, 32 of K a load, scores in powers of two.  32-bit: one, 16,
// natural exponentials, and products of 4x4x1 in sixteen blocks: a block is four weight rows and four rows of activations at one
// of the load's four places of K, so nothing is multiplied for rows that are not there (16x16x4 with four of its sixteen columns
// in use takes four times the clocks, 2.7 us an item at K of 3,072).
template <typename E> struct DcType;
template <> struct DcType<bf16_t> {
    static constexpr int PER_WORD = 2, STEP = 32;
    static __device__ __forceinline__ float exp(float x) { return fast_exp2(x); }
    static __device__ __forceinline__ bf16_t from(float v) { return f32_to_bf16(v); }
    // element e of a lane: weight row 4 (l/16) + e, row of activations l%16
    static __device__ __forceinline__ int x_row(int lane) { return lane & 15; }
    static __device__ __forceinline__ void multiply(dc_u32x4_t w, dc_u32x4_t x, f32x4_t& acc) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
    }
    static __device__ __forceinline__ void finish(f32x4_t&) {}
    static __device__ __forceinline__ int w_row(int lane) { return (lane >> 4) * 4; }
    static __device__ __forceinline__ bool holds(int lane, int rows) { return (lane & 15) < rows; }
};
template <> struct DcType<float> {
    static constexpr int PER_WORD = 1, STEP = 16;
    static __device__ __forceinline__ float exp(float x) { return expf(x); }
    static __device__ __forceinline__ float from(float v) { return v; }
    // element e of a lane: weight row 4 (l/4 % 4) + e, row of activations l%4, the places l/16 of K
    static __device__ __forceinline__ int x_row(int lane) { return lane & 3; }
    static __device__ __forceinline__ void multiply(dc_u32x4_t w, dc_u32x4_t x, f32x4_t& acc) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f32_4x4x1f32(__uint_as_float(w[e]), __uint_as_float(x[e]), acc, 0, 0, 0);
    }
    static __device__ __forceinline__ void finish(f32x4_t& acc) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[e] = rows4_sum(acc[e]);
        }
    }
    static __device__ __forceinline__ int w_row(int lane) { return (lane >> 2) * 4; }
    static __device__ __forceinline__ bool holds(int lane, int rows) { return lane < 16 && (lane & 3) < rows; }
};

struct DcLayer {
    const void *w_qkv, *w_o, *w_gu, *w_down;
    const float *q_gain, *k_gain;       // per-head norms
    const float* ffn_gain;              // the norm between attention and feed-forward
    const float* next_gain;             // the next layer's first norm (last layer: null)
    void *k, *v;                        // cache pages
};

// Word offsets of the buffers in the state (64-bit words).  The first DC_SHARDS lines hold the ticket counters, the next one the
// mark of a wait that gave up (dc_mark of its launch), the one behind it counts the blocks that have started.
struct DcPlan {
    int n_qkv, hq, hkv, hidden, inter, rows, splits, n_layers;
    int items[6], per_layer;            // work items of a layer's stages, in order
    int qkv_tiles, gu_tiles;            // tiles of an item of these stages
    int y, part, part_ml, o, xa, xga, ssqa, h, xb, xgb, ssqb, words;
    int waves, lds;
};

struct DcArgs {
    DcPlan p;
    u64* state;
    float* x;                           // [rows, hidden] residual stream, in and out
    const void* xn;                     // [rows, hidden] the first layer's normed operand
    const int* block_table; int bt_width;
    const int* pos;
    const float *cos_t, *sin_t;         // [rows, 64]
    float scale, qk_eps, eps_mix, eps_ffn, inv_width;
    int first_try;                      // what a wait's looks are counted from: 1 (a test looks at the clock earlier)
    long long patience;                 // DC_PATIENCE
    int* late;                          // host memory, or null: set to 1 when a wait gives up
    DcLayer layer[DC_LAYERS];
};

__device__ __forceinline__ u64 dc_load(const u64* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void dc_store(u64* p, uint32_t data, uint32_t epoch) {
    __hip_atomic_store(p, ((u64)epoch << 32) | data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What a launch leaves where a wait gave up, from the number that its words carry; never 0.
__device__ __forceinline__ u64 dc_mark(uint32_t epoch) { return (epoch - 2u) / (uint32_t)DC_LAYERS + 1u; }

// A wait that has gone on for long: true when it has to end, because this or another wait of the launch has lasted too long (a
// mark that an earlier launch left does not count).
__device__ __forceinline__ bool dc_give_up(const DcArgs& a, uint32_t epoch, int tries, u64& since) {
    if (tries & (DC_POLLS - 1)) return false;
    u64* at = a.state + DC_SHARDS * DC_LINE;
    if (since == 0) since = wall_clock64();
    if (dc_load(at) == dc_mark(epoch)) return true;
    if ((long long)(wall_clock64() - since) < a.patience) return false;
    __hip_atomic_store(at, dc_mark(epoch), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (a.late) __hip_atomic_store(a.late, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");          // (there before the NaN that the wait gives travels on)
    return true;
}

__device__ __forceinline__ const u64* dc_at(const u64* base, uint32_t bytes) { return (const u64*)((const char*)base + bytes); }

// N words a lane at the addresses that at(i, offset) gives, all of them of this epoch when it returns.  The whole wave stays
// until the last one is there.
template <int N, typename At>
__device__ __forceinline__ void dc_collect(const DcArgs& a, uint32_t epoch, bool mine, uint32_t offset, At at, uint32_t (&v)[N]) {
    u64 w[N], since = 0;
    for (int tries = a.first_try;; ++tries) {
        asm volatile("" : "+v"(offset));        // (the addresses are formed in every turn: they do not wait in registers)
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = dc_load(at(i, offset));
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) ok &= (uint32_t)(w[i] >> 32) == epoch;
        if (__all(ok || !mine)) break;
        if (dc_give_up(a, epoch, tries, since)) {
#pragma unroll
            for (int i = 0; i < N; ++i) w[i] = 0x7fc07fc0u;         // NaN, as one 32-bit number and as two of 16
            break;
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = (uint32_t)w[i];
}

// The block's first wave waits until one word of an earlier stage's result is there, asking now and then: until then nothing of
// what it waits for is near, and hundreds of blocks that ask for all their words all the time are in each other's way.
__device__ __forceinline__ void dc_far_wait(const DcArgs& a, const u64* word, uint32_t epoch) {
    u64 since = 0;
    for (int tries = a.first_try; (uint32_t)(__builtin_amdgcn_readfirstlane((int)(dc_load(word) >> 32))) != epoch; ++tries) {
        __builtin_amdgcn_s_sleep(16);
        if (dc_give_up(a, epoch, tries, since)) break;
    }
}

// 1 / sqrt(mean square of a row + eps) from the sums of squares of its tiles, of which the lane has added up its first two
// already; every lane gets it
__device__ __forceinline__ float dc_row_scale(const DcArgs& a, const u64* ssq, int tiles, uint32_t epoch, float eps, int lane,
                                              int from = 0, float ss = 0.f) {
    for (int at = from + lane; at - lane < tiles; at += 64) {       // (a word every DC_APART)
        uint32_t v[1];
        bool mine = at < tiles;
        dc_collect<1>(a, epoch, mine, mine ? at * (8u * DC_APART) : 0u, [&](int, uint32_t o) { return dc_at(ssq, o); }, v);
        ss += mine ? __uint_as_float(v[0]) : 0.f;
    }
    return 1.0f / sqrtf(wave_sum(ss) * a.inv_width + eps);
}

// A block's place in the order: {launch, ticket} of its counter, handed on as {launch, item}; the items shard, shard + DC_SHARDS,
// ... are the counter's.  A block draws until its ticket lies behind its counter's last item, so a counter is drawn from (items +
// blocks) times a launch; the last draw sets up the next launch.
struct DcTickets {
    u64* state; uint32_t end;           // the number behind the items that the counter's last draw gives; its counter is end % DC_SHARDS
    __device__ __forceinline__ u64* counter() const { return state + end % DC_SHARDS * DC_LINE; }
    __device__ __forceinline__ u64 draw() const { return __hip_atomic_fetch_add(counter(), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ __forceinline__ void drawn(u64 mine, u64* next) const {
        const uint32_t item = (uint32_t)mine * DC_SHARDS + end % DC_SHARDS;
        if (item == end) __hip_atomic_store(counter(), ((mine >> 32) + 1) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *next = (mine >> 32 << 32) | item;
    }
};

enum { DC_QKV = 0, DC_ATTN = 1, DC_MERGE = 2, DC_O = 3, DC_GU = 4, DC_DOWN = 5 };

template <int V> struct DcInt { static constexpr int value = V; };

// What a block works on, the same for all its threads.
struct DcItem { int stage, layer, i; uint32_t epoch; };

// LDS of a block.  (The arrays are read 16 bytes at a time; at an odd multiple of 8 a step takes a third longer.)
template <int W>
struct DcLds {
    u64 next[2];                                // the item after this one, in turn
    uint32_t end;                               // see DcTickets
    // The waves' sums, two of them in turn: behind an item's barrier its first waves (one for every four rows of its tiles, up to three)
    // read them while the others go on to the next item, which has the other place.  A place is written again two items later,
    // behind the barrier of the item between, which those waves reach when they have read.
    alignas(16) float red[2][DC_MAX_TILES][W][DC_MAX_ROWS][DC_TILE];
    float scale[2][DC_MAX_ROWS];                // the rows' norm scales, likewise
    alignas(16) float m[W][16], l[W][16];
    alignas(16) float o[W][DC_MAX_GROUP][DC_D + 4];
    alignas(16) float q[DC_MAX_GROUP][DC_D], k[DC_D], v[DC_D];      // (of the compute type)
    alignas(16) char x[];                       // operands of a product, rows of K values and DC_PAD bytes
};

__device__ __forceinline__ int dc_k(const DcPlan& p, int stage) { return stage == DC_O ? p.hq * DC_D : stage == DC_DOWN ? p.inter : p.hidden; }

// N rounds of 64 words of every row of operands (stride words apart) into LDS (pitch bytes apart), all asked for together.  SSQ:
// with them the first two rounds of the rows' sums of squares.
template <int M, int N, bool SSQ>
__device__ __forceinline__ void dc_take(const DcArgs& a, uint32_t epoch, const u64* row, int stride, char* to, int pitch, const u64* ssq, int tiles,
                                        int lane, float (&ss)[M]) {
    constexpr int E = SSQ ? 2 : 0;
    uint32_t v[M * (N + E)];
    dc_collect<M * (N + E)>(a, epoch, true, lane * 8u, [&](int i, uint32_t o) {
        const int m = i / (N + E), j = i % (N + E);
        return j < N ? dc_at(row + (size_t)m * stride + j * 64, o)
                     : dc_at(ssq + m * tiles * DC_APART, min(o + (j - N) * 512u, tiles * 8u - 8u) * DC_APART); }, v);
#pragma unroll
    for (int m = 0; m < M; ++m) {
        if constexpr (SSQ)
            ss[m] = (lane < tiles ? __uint_as_float(v[m * (N + E) + N]) : 0.f) + (lane + 64 < tiles ? __uint_as_float(v[m * (N + E) + N + 1]) : 0.f);
#pragma unroll
        for (int i = 0; i < N; ++i) *(uint32_t*)(to + m * pitch + (i * 64 + lane) * 4) = v[m * (N + E) + i];
    }
}

// SHORT: a wave's weights are all in its ring at once (separate code: one ring for both would be held twice).
// One to three tiles of 16 weight rows times all rows of activations.  A wave has an equal share of K: it asks for its weights, takes
// its share of the operands into LDS (nobody else reads it) and multiplies; the waves meet once, and the first ceil(tiles * rows / 4) of
// them finish, a row of lanes a tile of one row of activations.
__device__ __forceinline__ int dc_tiles(const DcPlan& p, int stage) { return stage == DC_QKV ? p.qkv_tiles : stage == DC_GU ? p.gu_tiles : 1; }

template <typename E, int W, int M, bool SHORT>
__device__ __forceinline__ void dc_product(const DcArgs& a, const DcLayer& ly, const DcItem& it, DcLds<W>& sm, const DcTickets& tickets, int turn,
                                           int wave, int lane) {
    using T = DcType<E>;
    constexpr int SIZE = sizeof(E), V = T::PER_WORD;
    const DcPlan& p = a.p;
    u64* st = a.state;
    const int stage = it.stage, layer = it.layer;
    const uint32_t epoch = it.epoch;
    const bool residual = stage == DC_O || stage == DC_DOWN, head = layer == 0;
    const int g = lane >> 4, col = lane & 15;
    const int tiles = SHORT ? dc_tiles(p, stage) : 1, tile0 = it.i * tiles;
    const E* w = (const E*)(stage == DC_QKV ? ly.w_qkv : stage == DC_O ? ly.w_o : stage == DC_GU ? ly.w_gu : ly.w_down);
    const int k = dc_k(p, stage), share = k / W, first = wave * share, groups = share / (T::STEP * DC_GROUP);
    auto strip = ga_buffer(w + (size_t)tile0 * DC_TILE * k, (long long)tiles * DC_TILE * k * SIZE);
    const uint32_t at = (uint32_t)(col * k + first) * SIZE + g * 16u;
    dc_u32x4_t ring[DC_RING][DC_GROUP];
    auto request = [&](int r, int group, int tile) {
        uint32_t from = group < groups && tile < tiles ? at : BUF_NOWHERE;
        uint32_t behind = (uint32_t)(tile * DC_TILE * k) * SIZE + group * (DC_GROUP * 64);
#pragma unroll
        for (int j = 0; j < DC_GROUP; ++j)
            ring[r][j] = __builtin_bit_cast(dc_u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(strip, from, behind + j * 64, 0));
    };
    {
        int group = 0, tile = 0;
#pragma unroll
        for (int r = 0; r < DC_RING; ++r) {
            request(r, group, tile);
            if (++group == groups && SHORT) { group = 0; ++tile; }
        }
    }
    // the first wave's lanes in the epilogue: a row of activations and one of 16 columns
    const int orow = lane >> 4, ocol = tile0 * DC_TILE + col;
    const bool mine = wave == 0 && orow < M;
    const float* gain = stage == DC_O ? ly.ffn_gain : ly.next_gain;
    float gv = 0.f, x_old = 0.f, ss[M];
#pragma unroll
    for (int m = 0; m < M; ++m) ss[m] = 0.f;
    if (residual && mine) {
        if (gain) gv = gain[ocol];
        if (stage == DC_O && head) x_old = a.x[(size_t)orow * p.hidden + ocol];
    }
    asm volatile("" ::: "memory");              // (the requests stay before the waits)
    __builtin_amdgcn_sched_barrier(0);
    const int pitch = k * SIZE + DC_PAD;
    // (the next item is drawn when this one's turn is near: drawn with the weights it would be bound to a block that still waits
    // while others have nothing to do, 37 against 30 us a layer; drawn at the end it would be waited for, 4 us a layer)
    u64 drawn = 0;
    if (stage == DC_QKV && head && wave == W - 1 && lane == 0) drawn = tickets.draw();
    if (stage == DC_QKV && head) {
#pragma unroll
        for (int m = 0; m < M; ++m)
            for (int i = lane; i < share / V; i += 64)
                *(uint32_t*)(sm.x + m * pitch + first * SIZE + i * 4) = ((const uint32_t*)((const E*)a.xn + (size_t)m * k + first))[i];
    } else {
        const u64* src = stage == DC_QKV ? st + p.xgb : stage == DC_O ? st + p.o : stage == DC_GU ? st + p.xga : st + p.h;
        const u64* far = stage == DC_QKV ? st + p.h : stage == DC_O ? st + p.y : stage == DC_GU ? st + p.o : st + p.xga;
        const int n_far = stage == DC_QKV ? p.inter / V : stage == DC_O ? p.n_qkv : stage == DC_GU ? p.hq * DC_D / V : p.hidden / V;
        const uint32_t src_epoch = stage == DC_QKV ? epoch - 1 : epoch;
        if (wave == 0) dc_far_wait(a, far + it.i * DC_LINE % n_far, src_epoch);
        __syncthreads();
        if (wave == W - 1 && lane == 0) drawn = tickets.draw();
        if (residual && wave == 0 && !(stage == DC_O && head)) {
            // (there before the operands are)
            uint32_t v[1];
            const u64* from = stage == DC_O ? st + p.xb : st + p.xa;
            dc_collect<1>(a, stage == DC_O ? epoch - 1 : epoch, mine, mine ? (uint32_t)(orow * p.hidden + ocol) * 8u : 0u,
                          [&](int, uint32_t o) { return dc_at(from, o); }, v);
            x_old = __uint_as_float(v[0]);
        }
        int left = share / (64 * V);
        const u64* row = src + first / V;
        char* to = sm.x + first * SIZE;
        auto take = [&](auto n, auto with_ssq) {
            constexpr int N = decltype(n)::value;
            dc_take<M, N, decltype(with_ssq)::value>(a, src_epoch, row, k / V, to, pitch, st + p.ssqa, p.hidden / DC_TILE, lane, ss);
            row += N * 64;
            to += N * 256;
            left -= N;
        };
        if (stage == DC_GU && wave == 0) {
            if (left >= 4) take(DcInt<4>{}, DcInt<1>{});
            else if (left >= 2) take(DcInt<2>{}, DcInt<1>{});
            else take(DcInt<1>{}, DcInt<1>{});
        }
        while (left >= 6) take(DcInt<6>{}, DcInt<0>{});
        if (left >= 4) take(DcInt<4>{}, DcInt<0>{});
        if (left >= 2) take(DcInt<2>{}, DcInt<0>{});
        if (left >= 1) take(DcInt<1>{}, DcInt<0>{});
    }
    if (wave == W - 1 && lane == 0) tickets.drawn(drawn, sm.next + (turn ^ 1));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();

    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const char* xs = sm.x + (M > 1 ? T::x_row(lane) % M : 0) * pitch + first * SIZE + g * 16;         // (columns beyond the rows repeat them)
    auto multiply = [&](int r, int group) {
        dc_u32x4_t xv[DC_GROUP];                // (read together: one by one each product waits for its own trip to LDS)
#pragma unroll
        for (int j = 0; j < DC_GROUP; ++j) xv[j] = *(const dc_u32x4_t*)(xs + (group * DC_GROUP + j) * 64);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < DC_GROUP; ++j)
            T::multiply(ring[r][j], xv[j], acc);
    };
    auto hand_over = [&](int tile) {
        T::finish(acc);
        if (T::holds(lane, M)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sm.red[turn][tile][wave][T::x_row(lane)][T::w_row(lane) + e] = acc[e];
        }
        acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    if constexpr (SHORT) {
        int group = 0, tile = 0;
#pragma unroll
        for (int r = 0; r < DC_RING; ++r) {
            if (tile < tiles) {
                multiply(r, group);
                if (++group == groups) {
                    hand_over(tile);
                    group = 0;
                    ++tile;
                }
            }
        }
    } else {
        for (int g0 = 0; g0 < groups; g0 += DC_RING) {
#pragma unroll
            for (int r = 0; r < DC_RING; ++r) {
                if (g0 + r < groups) multiply(r, g0 + r);
                request(r, g0 + r + DC_RING, 0);
            }
        }
        hand_over(0);
    }
    if (stage == DC_GU && wave == 0) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float scale = dc_row_scale(a, st + p.ssqa + m * (p.hidden / DC_TILE) * DC_APART, p.hidden / DC_TILE, epoch, a.eps_ffn, lane, 128, ss[m]);
            if (lane == 0) sm.scale[turn][m] = scale;
        }
    }
    __syncthreads();
    // A row of lanes finishes a tile of one row of activations: four of them a wave (one after the other in the first wave, the three
    // tiles of a gated item took a microsecond more).
    const int part = wave * 4 + g;
    if (wave * 4 >= tiles * M) return;
    const int row = part % M, tile = part / M;
    const bool in = tile < tiles;
    float v = 0.f;
    if (in) {
        const auto& red = sm.red[turn][tile];
        v = red[0][row][col];
#pragma unroll
        for (int i = 1; i < W; ++i) v += red[i][row][col];
    }
    if (stage == DC_QKV) {
        if (in) dc_store(st + p.y + (size_t)row * p.n_qkv + (tile0 + tile) * DC_TILE + col, __float_as_uint(v), epoch);
    } else if (stage == DC_GU) {
        // gate and up rows in turn: even lanes have a gate, their neighbour its up value
        v *= sm.scale[turn][row];
        const float up = lane_xor1(v), hv = v / (1.0f + expf(-v)) * up;
        u64* to = st + p.h + (size_t)row * (p.inter / V) + (tile0 + tile) * (8 / V);
        if constexpr (V == 2) {
            const float hn = lane_xor2(hv);
            if (in && (col & 3) == 0) dc_store(to + col / 4, f32x2_to_bf16x2(hv, hn), epoch);
        } else {
            if (in && (col & 1) == 0) dc_store(to + col / 2, __float_as_uint(hv), epoch);
        }
    } else {                                    // (one tile: the row is the one whose old value the lane holds)
        const float r = x_old + v;
        if (stage == DC_DOWN && layer == p.n_layers - 1) {
            if (in) a.x[(size_t)row * p.hidden + ocol] = r;
            return;
        }
        const float xg = r * gv, xn = lane_xor1(xg), sq = row16_sum(r * r);
        if (in) {
            const bool o = stage == DC_O;
            u64* to = st + (o ? p.xga : p.xgb) + (size_t)row * (p.hidden / V) + ocol / V;
            if (V == 1) dc_store(to, __float_as_uint(xg), epoch);
            else if ((col & 1) == 0) dc_store(to, f32x2_to_bf16x2(xg, xn), epoch);
            if (col == 0) dc_store(st + (o ? p.ssqa : p.ssqb) + (row * (p.hidden / DC_TILE) + tile0) * DC_APART, __float_as_uint(sq), epoch);
            dc_store(st + (o ? p.xa : p.xb) + (size_t)row * p.hidden + ocol, __float_as_uint(r), epoch);
        }
    }
}

// What the waves of an attention item do with the cached keys: the first piece is asked for before the projection is waited for
// (request_first), and behind the queries they multiply, their results meeting in LDS (run).
template <typename E, int W> struct DcPieces;

// bfloat16: a piece is 32 keys.
template <int W> struct DcPieces<bf16_t, W> {
    static constexpr int D = DC_D, KD = D / 32, DT = D / 16;
    const DcArgs& a; const DcLayer& ly; const int* pages;
    int kvh, split, my_pages, group, wave, lane;
    uint4 kbuf[2][KD], vbuf[DT];

    __device__ __forceinline__ void request(int piece) {
        const int g = lane >> 4, col = lane & 15;
        const size_t head = (size_t)pages[split + (piece >> 1) * a.p.splits] * a.p.hkv + kvh;
        const bf16_t* kb = (const bf16_t*)ly.k + (head * AM_PAGE + (piece & 1) * 32) * D;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int kd = 0; kd < KD; ++kd)
                kbuf[u][kd] = *(const uint4*)(kb + (uint32_t)((8 * (col >> 2) + 4 * u + (col & 3)) * D + g * 8 + kd * 32));
        const bf16_t* vb = (const bf16_t*)ly.v + head * D * AM_PAGE + (piece & 1) * 32;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vbuf[dt] = *(const uint4*)(vb + (uint32_t)((dt * 16 + col) * AM_PAGE + g * 8));
    }
    __device__ __forceinline__ void request_first() {
        if (wave < my_pages * 2) request(wave);
    }
    __device__ __forceinline__ void run(DcLds<W>& sm, bool owner, int new_pos) {
        const int g = lane >> 4, col = lane & 15, n_pieces = my_pages * 2;
        const float scale_log2e = a.scale * AM_LOG2E;
        const bf16_t *sq = (const bf16_t*)sm.q, *sk = (const bf16_t*)sm.k, *sv = (const bf16_t*)sm.v;
        // Q^T operand: column = head of the group (zero beyond it); read for every piece, registers are scarcer than LDS reads
        auto query = [&](int kd) {
            uint4 v = *(const uint4*)(sq + (col < group ? col : 0) * D + kd * 32 + g * 8);
            bool ok = col < group;
            v.x = ok ? v.x : 0u; v.y = ok ? v.y : 0u; v.z = ok ? v.z : 0u; v.w = ok ? v.w : 0u;
            return __builtin_bit_cast(bf16x8_t, v);
        };
        float m = -INFINITY, l = 0.f;
        f32x4_t o[DT];
#pragma unroll
        for (int i = 0; i < DT; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        auto scores = [&](int key0, int to, f32x4_t (&s)[2]) {
            // element i of s[u] is key 8g + 4u + i, column = head
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                s[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kd = 0; kd < KD; ++kd)
                    s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kbuf[u][kd]), query(kd), s[u], 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[u][i] = key0 + g * 8 + u * 4 + i < to ? s[u][i] * scale_log2e : -INFINITY;
        };
        auto add_values = [&](f32x4_t (&s)[2]) {
            float mx = -INFINITY;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[u][i]);
            mx = rows4_max(mx);
            float m_new = fmaxf(m, mx);
            float m_use = m_new == -INFINITY ? 0.f : m_new;
            float corr = fast_exp2(m - m_use), sum = 0.f;
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
            uint4 pv = make_uint4(pack_bf16x2(s[0][0], s[0][1]), pack_bf16x2(s[0][2], s[0][3]),
                                  pack_bf16x2(s[1][0], s[1][1]), pack_bf16x2(s[1][2], s[1][3]));
            bf16x8_t pf = __builtin_bit_cast(bf16x8_t, pv);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                o[dt] = o[dt] * corr;
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vbuf[dt]), pf, o[dt], 0, 0, 0);
            }
        };
        // (the step's own key is not yet in the cache where a block reads it: it takes its place in its piece from LDS)
        for (int piece = wave; piece < n_pieces; piece += W) {
            f32x4_t s[2];
            if (piece != wave) request(piece);
            const int key0 = (split + (piece >> 1) * a.p.splits) * AM_PAGE + (piece & 1) * 32, at = new_pos - key0;
            if (owner && at >= 0 && at < 32) {
                const bool krow = col == (at >> 3) * 4 + (at & 3);
                uint32_t half[4];                     // the value's half of a word of the lane's eight, if any
#pragma unroll
                for (int i = 0; i < 4; ++i) half[i] = g == at >> 3 && at % 8 / 2 == i ? (at & 1 ? 0xffff0000u : 0xffffu) : 0u;
#pragma unroll
                for (int kd = 0; kd < KD; ++kd) {
                    const uint4 v = *(const uint4*)(sk + kd * 32 + g * 8);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const bool take = krow && (at >> 2 & 1) == u;
                        uint4& k = kbuf[u][kd];
                        k = make_uint4(take ? v.x : k.x, take ? v.y : k.y, take ? v.z : k.z, take ? v.w : k.w);
                    }
                }
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const uint32_t v = sv[dt * 16 + col] * 0x10001u;
                    const uint4 old = vbuf[dt];
                    vbuf[dt] = make_uint4((old.x & ~half[0]) | (v & half[0]), (old.y & ~half[1]) | (v & half[1]),
                                          (old.z & ~half[2]) | (v & half[2]), (old.w & ~half[3]) | (v & half[3]));
                }
            }
            scores(key0, new_pos + 1, s);
            add_values(s);
        }
        // the waves' results in wave order; element i of o[dt] is d = 16 dt + 4g + i, column = head
        if (col < group) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) sm.o[wave][col][dt * 16 + g * 4 + i] = o[dt][i];
        }
        if (g == 0) {
            sm.m[wave][col] = m;
            sm.l[wave][col] = l;
        }
    }
};

// 32-bit: a piece is 16 keys, multiplied as the projections are (4x4x1 in sixteen blocks, four heads at a time): a block is four keys and four heads
// at one place of the head size, or four values and four heads at one key, and the four rows of lanes add up.  16x16x4 with the two heads of a
// group in use takes four times the clocks: 2 us a piece.
template <int W> struct DcPieces<float, W> {
    static constexpr int D = DC_D, KD = D / 16, HEADS = (DC_MAX_GROUP + 3) / 4;
    const DcArgs& a; const DcLayer& ly; const int* pages;
    int kvh, split, my_pages, group, wave, lane;
    af_f32x4_t k[KD], v[KD];

    __device__ __forceinline__ void request(int piece) {
        const size_t at = ((size_t)pages[split + (piece >> 2) * a.p.splits] * a.p.hkv + kvh) * AF_PAGE * D;
        const int in_page = (piece & 3) * 16;
        const float* kp = (const float*)ly.k + at + (uint32_t)((in_page + (lane & 15)) * D + (lane >> 4) * 4);
        const float* vp = (const float*)ly.v + at + (uint32_t)((lane & 15) * AF_PAGE + in_page + (lane >> 4) * 4);
#pragma unroll
        for (int c = 0; c < KD; ++c) k[c] = *(const af_f32x4_t*)(kp + c * 16);
#pragma unroll
        for (int c = 0; c < KD; ++c) v[c] = *(const af_f32x4_t*)(vp + c * 16 * AF_PAGE);
    }
    __device__ __forceinline__ void request_first() {
        if (wave < my_pages * 4) request(wave);
    }
    __device__ __forceinline__ void run(DcLds<W>& sm, bool owner, int new_pos) {
        const int n_pieces = my_pages * 4, g = lane >> 4, quad = lane >> 2 & 3;
        af_f32x4_t o[HEADS][KD];
        float m[HEADS], l[HEADS];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            m[h] = -INFINITY;
            l[h] = 0.f;
#pragma unroll
            for (int c = 0; c < KD; ++c) o[h][c] = af_f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        for (int piece = wave; piece < n_pieces; piece += W) {
            const int first = (split + (piece >> 2) * a.p.splits) * AF_PAGE + (piece & 3) * 16, at = new_pos - first;
            if (at < 0) continue;
            if (piece != wave) request(piece);
            // (the step's own key is not yet in the cache where a block reads it: it takes its place in its piece from LDS; a key that is
            // not seen may hold anything: it is left out, not weighted by zero)
            const bool own = owner && at < 16;
            if (own) {
#pragma unroll
                for (int c = 0; c < KD; ++c) {
                    const af_f32x4_t nk = *(const af_f32x4_t*)(sm.k + c * 16 + g * 4);
                    const float nv = sm.v[c * 16 + (lane & 15)];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        k[c][e] = (lane & 15) == at ? nk[e] : k[c][e];
                        v[c][e] = g * 4 + e == at ? nv : v[c][e];
                    }
                }
            }
            if (at < 15) {
#pragma unroll
                for (int c = 0; c < KD; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[c][e] = g * 4 + e <= at ? v[c][e] : 0.f;
            }
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                if (h * 4 >= group) break;
                const float* q = sm.q[min(h * 4 + (lane & 3), group - 1)] + g * 4;
                f32x4_t s = {0.f, 0.f, 0.f, 0.f}, odd = s;
#pragma unroll
                for (int c = 0; c < KD; ++c) {
                    const af_f32x4_t qv = *(const af_f32x4_t*)(q + c * 16);
#pragma unroll
                    for (int e = 0; e < 4; e += 2) {
                        s = __builtin_amdgcn_mfma_f32_4x4x1f32(k[c][e], qv[e], s, 0, 0, 0);
                        odd = __builtin_amdgcn_mfma_f32_4x4x1f32(k[c][e + 1], qv[e + 1], odd, 0, 0, 0);
                    }
                }
                // element e: key 4 quad + e, head l%4, the same in every row of lanes
                float top = -INFINITY;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float sum = rows4_sum(s[e] + odd[e]) * a.scale;       // (by all lanes, seen or not)
                    s[e] = quad * 4 + e <= at ? sum : -INFINITY;
                    top = fmaxf(top, s[e]);
                }
                top = fmaxf(top, lane_dpp<0x128>(top));             // (rotated by 8 and by 4 lanes inside the row)
                top = fmaxf(top, lane_dpp<0x124>(top));
                const float m_new = fmaxf(m[h], top), ref = m_new == -INFINITY ? 0.f : m_new, corr = expf(m[h] - ref);
                l[h] *= corr;
                af_f32x4_t p;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[e] = expf(s[e] - ref);
                    l[h] += s[e];
                    p[e] = __shfl(s[e], g * 20 + (lane & 3), 64);    // key 4 (l/16) + e: of this row's quad of that number
                }
                m[h] = m_new;
#pragma unroll
                for (int c = 0; c < KD; ++c) o[h][c] *= corr;
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < KD; ++c) o[h][c] = __builtin_amdgcn_mfma_f32_4x4x1f32(v[c][e], p[e], o[h][c], 0, 0, 0);
            }
        }
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            if (h * 4 >= group) break;
            const int row = h * 4 + (lane & 3);
            l[h] += lane_dpp<0x128>(l[h]);
            l[h] += lane_dpp<0x124>(l[h]);
            if (lane < 4) {
                sm.m[wave][row] = m[h];
                sm.l[wave][row] = l[h];
            }
#pragma unroll
            for (int c = 0; c < KD; ++c) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[h][c][e] = rows4_sum(o[h][c][e]);
                if (g == 0 && row < group) *(af_f32x4_t*)(&sm.o[wave][row][c * 16 + quad * 4]) = o[h][c];
            }
        }
    }
};

// Two neighbouring values of a (token, head)'s output.
template <typename E>
__device__ __forceinline__ void dc_store_pair(u64* out, int row, int lane, float v0, float v1, uint32_t epoch) {
    if constexpr (DcType<E>::PER_WORD == 2) {
        dc_store(out + (size_t)row * (DC_D / 2) + lane, f32x2_to_bf16x2(v0, v1), epoch);
    } else {
        dc_store(out + (size_t)row * DC_D + lane * 2, __float_as_uint(v0), epoch);
        dc_store(out + (size_t)row * DC_D + lane * 2 + 1, __float_as_uint(v1), epoch);
    }
}

// One (token, kv head, split of its pages): the query heads of the kv head from the projection, the cached keys, and in the
// block whose split holds the last page the step's own key and value, which it also appends.  Pages split, split + splits, ...;
// the waves take their pieces in turn.
template <typename E, int W>
__device__ __forceinline__ void dc_attention(const DcArgs& a, const DcLayer& ly, const DcItem& it, DcLds<W>& sm, const DcTickets& tickets, int turn,
                                             int wave, int lane) {
    constexpr int D = DC_D, ROWS = (DC_MAX_GROUP + 2 + W - 1) / W;
    using T = DcType<E>;
    const DcPlan& p = a.p;
    u64* st = a.state;
    const uint32_t epoch = it.epoch;
    const int g = lane >> 4, col = lane & 15;
    const int split = it.i % p.splits, kvh = it.i / p.splits % p.hkv, t = it.i / (p.splits * p.hkv);
    const int group = p.hq / p.hkv;
    const int* pages = a.block_table + (size_t)t * a.bt_width;
    const int new_pos = a.pos[t], len = new_pos + 1;
    const int n_pages = (len + AM_PAGE - 1) / AM_PAGE;
    const int my_pages = split < n_pages ? (n_pages - split + p.splits - 1) / p.splits : 0;
    DcPieces<E, W> piece{a, ly, pages, kvh, split, my_pages, group, wave, lane};
    piece.request_first();
    const bool owner = new_pos / AM_PAGE % p.splits == split;
    const int phys = pages[new_pos / AM_PAGE];
    const int n_rows = group + (owner ? 2 : 0);
    const float cs = a.cos_t[t * (D / 2) + lane], si = a.sin_t[t * (D / 2) + lane];
    const float gq0 = ly.q_gain[lane], gq1 = ly.q_gain[lane + 64], gk0 = ly.k_gain[lane], gk1 = ly.k_gain[lane + 64];
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    float row_scale = 1.0f;
    if (it.layer > 0) {
        if (wave == 0) dc_far_wait(a, st + p.xgb + it.i * DC_LINE % (p.hidden / T::PER_WORD), epoch - 1);
        __syncthreads();
        row_scale = dc_row_scale(a, st + p.ssqb + t * (p.hidden / DC_TILE) * DC_APART, p.hidden / DC_TILE, epoch - 1, a.eps_mix, lane);
    }
    u64 drawn = 0;
    if (wave == W - 1 && lane == 0) drawn = tickets.draw();
    // a wave's rows of the projection together: a lane has the values lane and lane + 64 of each
    {
        const u64* tok = st + p.y + (size_t)t * p.n_qkv;
        auto from = [&](int r) { return tok + (size_t)(r < group ? kvh * group + r : r == group ? p.hq + kvh : p.hq + p.hkv + kvh) * D; };
        uint32_t raw[2 * ROWS];
        dc_collect<2 * ROWS>(a, epoch, true, lane * 8u, [&](int i, uint32_t o) {
            return dc_at(from(min(wave + i / 2 * W, n_rows - 1)) + (i & 1) * 64, o); }, raw);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            int r = wave + W * i;
            if (r >= n_rows) break;
            float v0 = __uint_as_float(raw[2 * i]) * row_scale, v1 = __uint_as_float(raw[2 * i + 1]) * row_scale;
            if (r <= group) {
                float inv = 1.0f / sqrtf(wave_sum(fmaf(v1, v1, v0 * v0)) / (float)D + a.qk_eps);
                v0 = v0 * inv * (r < group ? gq0 : gk0);
                v1 = v1 * inv * (r < group ? gq1 : gk1);
                // pairs (e, e + 64) are one lane's
                float lo = v0 * cs - v1 * si, hi = v0 * si + v1 * cs;
                v0 = lo;
                v1 = hi;
            }
            E b0 = T::from(v0), b1 = T::from(v1);
            E* dst = r < group ? (E*)sm.q + r * D : r == group ? (E*)sm.k : (E*)sm.v;
            dst[lane] = b0;
            dst[lane + 64] = b1;
            // (what a wait that gave up has made of a key or value stays out of the cache: a page's next sequence may weight the
            // row by zero, which does not take a NaN away)
            const bool lost = r >= group && __any(v0 != v0 || v1 != v1) && dc_load(st + DC_SHARDS * DC_LINE) == dc_mark(epoch);
            if (phys >= 0 && r >= group && !lost) {
                const size_t head = (size_t)phys * p.hkv + kvh;
                const int at = new_pos % AM_PAGE;
                if (r == group) {
                    ((E*)ly.k)[(head * AM_PAGE + at) * D + lane] = b0;
                    ((E*)ly.k)[(head * AM_PAGE + at) * D + lane + 64] = b1;
                } else {
                    ((E*)ly.v)[(head * D + lane) * AM_PAGE + at] = b0;
                    ((E*)ly.v)[(head * D + lane + 64) * AM_PAGE + at] = b1;
                }
            }
        }
    }
    if (wave == W - 1 && lane == 0) tickets.drawn(drawn, sm.next + (turn ^ 1));
    __syncthreads();
    piece.run(sm, owner, new_pos);
    __syncthreads();
    for (int head = wave; head < group; head += W) {
        const int d = lane * 2;
        float mm = sm.m[0][head];
#pragma unroll
        for (int w = 1; w < W; ++w) mm = fmaxf(mm, sm.m[w][head]);
        float ll = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            float wgt = sm.m[w][head] == -INFINITY ? 0.f : T::exp(sm.m[w][head] - mm);
            ll += sm.l[w][head] * wgt;
            o0 += sm.o[w][head][d] * wgt;
            o1 += sm.o[w][head][d + 1] * wgt;
        }
        int row = t * p.hq + kvh * group + head;
        if (p.splits == 1) {
            dc_store_pair<E>(st + p.o, row, lane, o0 / ll, o1 / ll, epoch);
        } else {
            size_t slot = (size_t)row * p.splits + split;
            dc_store(st + p.part + slot * D + d, __float_as_uint(o0), epoch);
            dc_store(st + p.part + slot * D + d + 1, __float_as_uint(o1), epoch);
            if (lane == 0) {
                dc_store(st + p.part_ml + slot * 2, __float_as_uint(mm), epoch);
                dc_store(st + p.part_ml + slot * 2 + 1, __float_as_uint(ll), epoch);
            }
        }
    }
    __syncthreads();                            // (the LDS is the next item's)
}

// The splits of one (token, query head) by log-sum-exp in split order, a run of them a wave.
template <typename E, int W>
__device__ __forceinline__ void dc_merge(const DcArgs& a, const DcItem& it, DcLds<W>& sm, const DcTickets& tickets, int turn, int wave, int lane) {
    constexpr int D = DC_D;
    const DcPlan& p = a.p;
    u64* st = a.state;
    const uint32_t epoch = it.epoch;
    const int row = it.i;
    if (wave == 0) dc_far_wait(a, st + p.y + row * DC_LINE % p.n_qkv, epoch);
    __syncthreads();
    u64 drawn = 0;
    if (wave == W - 1 && lane == 0) drawn = tickets.draw();
    const u64* ml = st + p.part_ml + (size_t)row * p.splits * 2;
    bool mine = lane < p.splits;
    uint32_t v[2];
    dc_collect<2>(a, epoch, mine, mine ? lane * 16u : 0u, [&](int i, uint32_t o) { return dc_at(ml + i, o); }, v);
    float ms = mine ? __uint_as_float(v[0]) : -INFINITY, ls = mine ? __uint_as_float(v[1]) : 0.f;
    float mm = wave_max(ms);
    float wgt = ms == -INFINITY ? 0.f : DcType<E>::exp(ms - mm);
    float inv_l = 1.0f / wave_sum(ls * wgt);    // every wave computes the same sum
    const int run = (p.splits + W - 1) / W, s1 = min(p.splits, (wave + 1) * run);
    float o0 = 0.f, o1 = 0.f;
    for (int s0 = wave * run; s0 < s1; s0 += 4) {
        uint32_t q[8];
        dc_collect<8>(a, epoch, true, lane * 8u, [&](int i, uint32_t o) {
            return dc_at(st + p.part + ((size_t)row * p.splits + min(s0 + i / 2, s1 - 1)) * D + (i & 1) * 64, o); }, q);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float ws = s0 + i < s1 ? __shfl(wgt, s0 + i, 64) : 0.f;
            o0 += __uint_as_float(q[2 * i]) * ws;
            o1 += __uint_as_float(q[2 * i + 1]) * ws;
        }
    }
    sm.o[wave][0][lane] = o0;
    sm.o[wave][0][lane + 64] = o1;
    if (wave == W - 1 && lane == 0) tickets.drawn(drawn, sm.next + (turn ^ 1));
    __syncthreads();
    if (wave == 0) {
        float r[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int d = lane * 2 + j;
            float sum = sm.o[0][0][d];
#pragma unroll
            for (int i = 1; i < W; ++i) sum += sm.o[i][0][d];
            r[j] = sum * inv_l;
        }
        dc_store_pair<E>(st + p.o, row, lane, r[0], r[1], epoch);
    }
    __syncthreads();                            // (the LDS is the next item's)
}

template <typename E, int W, int M>
__global__ void __launch_bounds__(64 * W) decode_chain_kernel(const DcArgs a) {
    extern __shared__ __attribute__((aligned(16))) char dc_lds[];
    DcLds<W>& sm = *(DcLds<W>*)dc_lds;
    const DcPlan& p = a.p;
    const uint32_t total = (uint32_t)p.per_layer * p.n_layers;
    if (threadIdx.x == 0) {
        // (a launch's blocks are a whole number for every counter, so the count goes on from launch to launch)
        const u64 started = __hip_atomic_fetch_add(a.state + (DC_SHARDS + 1) * DC_LINE, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t shard = (uint32_t)(started % DC_SHARDS);
        sm.end = ((total - shard + DC_SHARDS - 1) / DC_SHARDS + gridDim.x / DC_SHARDS - 1) * DC_SHARDS + shard;
        const DcTickets mine = {a.state, sm.end};
        mine.drawn(mine.draw(), sm.next);
    }
    __syncthreads();
    uint32_t end = sm.end;
    // (a vector register: scalar ones are scarcer.  1 % of a step of 530 us when it was measured, before stages and layers were in scalar
    // registers too)
    asm volatile("" : "+v"(end));
    const DcTickets tickets = {a.state, end};
    for (int turn = 0;; turn ^= 1) {
        const u64 drawn = sm.next[turn];
        const uint32_t item = __builtin_amdgcn_readfirstlane((int)(uint32_t)drawn);
        const uint32_t launch = __builtin_amdgcn_readfirstlane((int)(uint32_t)(drawn >> 32));
        if (item >= total) break;
        DcItem it;
        it.layer = item / p.per_layer;
        it.i = item - it.layer * p.per_layer;
        it.stage = 0;
#pragma unroll
        for (int s = 0; s < 5; ++s)
            if (it.stage == s && it.i >= p.items[s]) {
                it.i -= p.items[s];
                it.stage = s + 1;
            }
        // (told to be the same in all lanes: the divisions leave them in vector registers, and a choice between two operands by the
        // stage was then a load of the kernel's arguments by the lanes and a wait for everything on its way, the last store included: 1 to
        // 2 us in every output and down item)
        it.layer = __builtin_amdgcn_readfirstlane(it.layer);
        it.i = __builtin_amdgcn_readfirstlane(it.i);
        it.stage = __builtin_amdgcn_readfirstlane(it.stage);
        // (numbers start at 2: the state starts as zeros, and a layer reads what the one before it numbered)
        it.epoch = launch * (uint32_t)DC_LAYERS + (uint32_t)it.layer + 2u;
        const DcLayer& ly = a.layer[it.layer];
        // (told to be new in every turn: what the stages derive from it is not kept in registers beside the weights)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        if (it.stage == DC_ATTN) dc_attention<E, W>(a, ly, it, sm, tickets, turn, wave, lane);
        else if (it.stage == DC_MERGE) dc_merge<E, W>(a, it, sm, tickets, turn, wave, lane);
        else if (dc_tiles(p, it.stage) * dc_k(p, it.stage) <= DC_RING * DC_GROUP * DcType<E>::STEP * W)
            dc_product<E, W, M, true>(a, ly, it, sm, tickets, turn, wave, lane);
        else dc_product<E, W, M, false>(a, ly, it, sm, tickets, turn, wave, lane);
    }
}

// Whether a layer's sizes fit, and the plan of buffers and blocks (words of 64 bits).
static bool dc_plan(DcPlan& p, int dtype, int rows, int hidden, int hq, int hkv, int head_dim, int inter, int n_layers, int splits) {
    if (rows < 1 || rows > DC_MAX_ROWS || head_dim != DC_D || hkv < 1 || hq < hkv || hq % hkv != 0 || hq / hkv > DC_MAX_GROUP) return false;
    if (n_layers < 1 || n_layers > DC_LAYERS || splits < 1 || splits > 64) return false;
    // a wave's share of K in whole groups of steps; strips of 16 weight rows whose offsets fit 31 bits
    if (dtype != ROCML_BF16 && dtype != ROCML_F32) return false;
    const bool f32 = dtype == ROCML_F32;
    // 32-bit and wide layers: eight waves a block, so that a wave's share of K fits its ring (1.7B, one row: 500 -> 455 us a step;
    // 0.6B in bfloat16, whose shares fit four waves' rings, 548 -> 648)
    p.waves = f32 || (hidden >= 2048 && hidden % 1024 == 0 && inter % 1024 == 0 && hq * DC_D % 1024 == 0) ? 8 : 4;
    const int unit = (f32 ? 16 : 32) * DC_GROUP * p.waves, v = f32 ? 1 : 2, size = f32 ? 4 : 2;
    if (hidden < unit || inter < unit || hidden % unit != 0 || inter % unit != 0 || hq * (long long)DC_D % unit != 0) return false;
    if (hidden > (1 << 20) || inter > (1 << 20) || hq > (1 << 13)) return false;
    p.rows = rows; p.hidden = hidden; p.hq = hq; p.hkv = hkv; p.inter = inter; p.n_layers = n_layers; p.splits = splits;
    p.n_qkv = (hq + 2 * hkv) * DC_D;
    // short K: several tiles an item, as many as a wave's ring of weights holds (0.6B: 392 items a layer instead of 776)
    auto tiles = [&](int n_tiles) {
        const int groups = hidden / unit;
        for (int t = DC_MAX_TILES; t > 1; --t)
            if (t * groups <= DC_RING && n_tiles % t == 0) return t;
        return 1;
    };
    p.qkv_tiles = tiles(p.n_qkv / DC_TILE);
    p.gu_tiles = tiles(2 * inter / DC_TILE);
    p.items[DC_QKV] = p.n_qkv / DC_TILE / p.qkv_tiles;
    p.items[DC_ATTN] = rows * hkv * splits;
    p.items[DC_MERGE] = splits > 1 ? rows * hq : 0;
    p.items[DC_O] = hidden / DC_TILE;
    p.items[DC_GU] = 2 * inter / DC_TILE / p.gu_tiles;
    p.items[DC_DOWN] = hidden / DC_TILE;
    p.per_layer = 0;
    for (int s = 0; s < 6; ++s) p.per_layer += p.items[s];
    int at = (DC_SHARDS + 2) * DC_LINE;
    auto take = [&](long long words) { int here = at; at += (int)((words + 15) / 16 * 16); return here; };
    p.y = take((long long)rows * p.n_qkv);
    p.part = take(splits > 1 ? (long long)rows * hq * splits * DC_D : 0);
    p.part_ml = take(splits > 1 ? (long long)rows * hq * splits * 2 : 0);
    p.o = take((long long)rows * hq * DC_D / v);
    p.xa = take((long long)rows * hidden); p.xb = take((long long)rows * hidden);
    p.xga = take((long long)rows * hidden / v); p.xgb = take((long long)rows * hidden / v);
    p.ssqa = take((long long)rows * hidden / DC_TILE * DC_APART); p.ssqb = take((long long)rows * hidden / DC_TILE * DC_APART);
    p.h = take((long long)rows * inter / v);
    p.words = at;
    const int most_k = inter > hidden ? (inter > hq * DC_D ? inter : hq * DC_D) : (hidden > hq * DC_D ? hidden : hq * DC_D);
    const long long product = (long long)rows * (most_k * (long long)size + DC_PAD);
    const long long lds = (p.waves == 8 ? sizeof(DcLds<8>) : sizeof(DcLds<4>)) + product;
    if (lds > DC_MAX_LDS) return false;
    p.lds = (int)lds;
    return true;
}

// The most pages of a step's block table with which the chain is faster than the layers' own kernels; 0: never.  A matter of how
// long the weights' bytes take beside the stages' latencies, of how many words travel, and of how many keys are seen: the attention
// kernels have a piece of keys on its way while they multiply another, the chain, whose registers hold weights, has not.  Steps to
// the logits, replayed, us:
//   bfloat16, 0.6B (31 MB a layer), one row: 40 keys 1,002 -> 474, 5,000 1,094 -> 703, 20,000 1,350 -> 1,228, 40,000 (626 pages) 1,724 -> 1,781; two rows: 2,000
//     1,003 -> 650, 8,000 1,323 -> 1,101, 16,000 (251 pages) 1,601 -> 1,531; three: 2,100 1,162 -> 871, 4,000 1,287 -> 1,051; four: 2,100 1,227 -> 967, 4,000
//     1,362 -> 1,195, 8,000 (126 pages) 1,654 -> 1,674;
//   1.7B (100 MB, 8 layers), one row: 500 523 -> 391, 32,000 701 -> 684; two: 4,200 562 -> 515, 8,000 604 -> 572; four: 500 551 -> 489, 4,000 628 -> 601;
//   4B (202 MB, 6 layers): one row 608 -> 597, four 641 -> 711; 8B (386 MB, 6 layers): one 806 -> 802, two 818 -> 845: while weights stream, a word's way takes several us;
//   32-bit, whose attention kernels walk a sequence's keys in few blocks: 0.6B (63 MB), one row of 5,000 6,039 -> 1,187, four of 300 1,703 -> 1,016,
//     of 4,000 5,210 -> 1,817; 1.7B (201 MB), one row of 500 962 -> 774, two 976 -> 804 (four do not fit the LDS).
// The lines for several rows, and one row for large 32-bit layers, were drawn when the chain was slower; tests/test_gpu_decode_chain.py holds
// them.  By the figures above they could lie at 250 pages for two rows and some 110 for four.
ROCML_EXPORT int rocml_decode_chain_reach(int dtype, int rows, int hidden, int hq, int hkv, int head_dim, int inter) {
    DcPlan p;
    if (!dc_plan(p, dtype, rows, hidden, hq, hkv, head_dim, inter, 1, 1)) return 0;
    const double mb = (dtype == ROCML_F32 ? 4e-6 : 2e-6) * hidden * ((double)p.n_qkv + (double)hq * DC_D + 3.0 * inter);
    if (mb > (dtype == ROCML_F32 && rows == 1 ? 256.0 : 128.0)) return 0;
    return dtype == ROCML_F32 ? 0x7fffffff : rows == 1 ? 512 : 128 / rows;
}

// 64-bit words of state that a chain of such layers needs; 0: not taken.
ROCML_EXPORT int rocml_decode_chain_words(int dtype, int rows, int hidden, int hq, int hkv, int head_dim, int inter, int n_layers, int splits) {
    DcPlan p;
    return dc_plan(p, dtype, rows, hidden, hq, hkv, head_dim, inter, n_layers, splits) ? p.words : 0;
}

ROCML_EXPORT int rocml_decode_chain_max_layers() { return DC_LAYERS; }

// layers: per layer the ten pointers of DcLayer.  polls (looks before a wait's first look at the clock), patience (ticks of
// 10 ns): when a wait gives up; 0 and -1: as it is meant.  late: see DcArgs.  blocks: 0 for a block a CU; at least so many are started, and eight do.
ROCML_EXPORT int rocml_decode_chain(int dtype, void* state, long long state_words, float* x, const void* xn, const void* const* layers, int n_layers,
                                    int rows, int hidden, int hq, int hkv, int head_dim, int inter, const int* block_table, int bt_width,
                                    const int* token_pos, const float* cos_t, const float* sin_t, float scale, float qk_eps, float eps_mix,
                                    float eps_ffn, int splits, int polls, long long patience, int* late, int blocks,
                                    hipStream_t stream) {
    DcArgs a;
    ROCML_REQUIRE(dc_plan(a.p, dtype, rows, hidden, hq, hkv, head_dim, inter, n_layers, splits),
                  "decode_chain: sizes not taken: rows=%d hidden=%d heads=%d/%d of %d inter=%d layers=%d splits=%d", rows, hidden, hq, hkv,
                  head_dim, inter, n_layers, splits);
    ROCML_REQUIRE(state && state_words >= a.p.words, "decode_chain: the state has %lld of %d words", state_words, a.p.words);
    ROCML_REQUIRE(x && xn && layers && block_table && token_pos && cos_t && sin_t && bt_width > 0, "decode_chain: missing operand");
    ROCML_REQUIRE(polls >= 0 && polls <= DC_POLLS, "decode_chain: %d looks", polls);
    a.first_try = polls > 0 ? DC_POLLS + 1 - polls : 1;
    a.patience = patience >= 0 ? patience : DC_PATIENCE;
    a.late = late;
    a.state = (u64*)state;
    a.x = x; a.xn = xn; a.block_table = block_table; a.bt_width = bt_width; a.pos = token_pos;
    a.cos_t = cos_t; a.sin_t = sin_t;
    a.scale = scale; a.qk_eps = qk_eps; a.eps_mix = eps_mix; a.eps_ffn = eps_ffn; a.inv_width = 1.0f / (float)hidden;
    for (int i = 0; i < n_layers; ++i) {
        const void* const* f = layers + 10 * i;
        for (int j = 0; j < 10; ++j) ROCML_REQUIRE(f[j] || (j == 7 && i == n_layers - 1), "decode_chain: layer %d lacks operand %d", i, j);
        for (int j : {0, 1, 2, 3, 8, 9}) ROCML_REQUIRE((uintptr_t)f[j] % 16 == 0, "decode_chain: operand %d of layer %d is not aligned", j, i);
        a.layer[i] = DcLayer{f[0], f[1], f[2], f[3], (const float*)f[4], (const float*)f[5], (const float*)f[6], (const float*)f[7],
                             (void*)f[8], (void*)f[9]};
    }
    // a block a CU; a whole number for every counter
    ROCML_REQUIRE(blocks >= 0, "decode_chain: %d blocks", blocks);
    blocks = ceil_div(blocks > 0 ? blocks : cu_count(), DC_SHARDS) * DC_SHARDS;
    typedef void (*Kernel)(DcArgs);
    static const Kernel kernels[3][DC_MAX_ROWS] = {
        {decode_chain_kernel<float, 8, 1>, decode_chain_kernel<float, 8, 2>, decode_chain_kernel<float, 8, 3>, decode_chain_kernel<float, 8, 4>},
        {decode_chain_kernel<bf16_t, 4, 1>, decode_chain_kernel<bf16_t, 4, 2>, decode_chain_kernel<bf16_t, 4, 3>, decode_chain_kernel<bf16_t, 4, 4>},
        {decode_chain_kernel<bf16_t, 8, 1>, decode_chain_kernel<bf16_t, 8, 2>, decode_chain_kernel<bf16_t, 8, 3>, decode_chain_kernel<bf16_t, 8, 4>}};
    const Kernel kernel = kernels[dtype == ROCML_F32 ? 0 : a.p.waves == 4 ? 1 : 2][rows - 1];
    if (a.p.lds > (64 << 10))
        ROCML_REQUIRE(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, DC_MAX_LDS) == hipSuccess,
                      "decode_chain: %d bytes of LDS were refused", a.p.lds);
    kernel<<<blocks, 64 * a.p.waves, a.p.lds, stream>>>(a);
    ROCML_CHECK_LAUNCH("decode_chain");
    return 0;
}
