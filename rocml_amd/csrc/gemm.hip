// Matrix products of the decoder: out[M,N] (+)= X[M,K] * W[N,K]^T, weights row-major
// [out, in] as the reference keeps them (rocml/src/weights/mod.rs:78-98).  bfloat16 operands
// go to the MFMA kernels and 32-bit operands to the 32-bit matrix instructions (gemm_f32.h) when
// their layout allows 16-byte loads; everything else goes to the plain tiled kernel.
#include "common.h"
#include "gemm_tile.h"
#include "gemm_mfma.h"
#include "gemm_pingpong.h"
#include "gemm_ring.h"

ROCML_LAST_ERROR_FN(gemm)

// (the tile kernels by rows x columns of a block's tile)
enum GemmAlgo : int { ALGO_AUTO = 0, ALGO_PLAIN = 1, ALGO_MFMA_TILE = 2, ALGO_MFMA_SKINNY = 3, ALGO_MFMA_KPAR = 4,
                      ALGO_MFMA_TILE256 = 5, ALGO_MFMA_TILE256X192 = 6, ALGO_MFMA_TILE128X192 = 7, ALGO_MFMA_TILE256X128 = 8,
                      ALGO_MFMA_TILE64X128 = 9, ALGO_MFMA_TILE64 = 10, ALGO_MFMA_TILE128X64 = 11, ALGO_MFMA_TILE128X256 = 12 };

static int round_up(int a, int b) { return (a + b - 1) / b * b; }

template <typename K>
static int allow_lds(K kernel, int bytes, const char* name) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess)
        return rocml_fail("%s: cannot reserve %d bytes of LDS: %s", name, bytes, hipGetErrorString(e));
    return 0;
}

struct SplitPlan { int defer; int* deferred; RowScale rs; int max_splits; };   // max_splits: the most K pieces the caller wants

template <int EPI, typename T, typename E = bf16_t>
static int launch_mfma_tile_as(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m,
                               int n, int k, int splits, void* workspace, SplitPlan plan, hipStream_t stream) {
    static bool ready = false;
    if (!ready) {
        if (allow_lds(gemm_mfma_kernel<EPI, T, E>, T::LDS_BYTES, "gemm")) return 1;
        if (allow_lds(gemm_mfma_kernel<EPI_F32, T, E>, T::LDS_BYTES, "gemm")) return 1;
        ready = true;
    }
    int tiles_m = ceil_div(m, T::BM), tiles_n = ceil_div(n, T::BN);
    int n_tiles = tiles_m * tiles_n;
    if (splits <= 1) {
        gemm_mfma_kernel<EPI, T, E><<<round_up(n_tiles, 8), T::THREADS, T::LDS_BYTES, stream>>>(
            (const E*)x, ldx, (const E*)w, ldw, out, ldo, m, n, k, tiles_m, n_tiles, k, 0);
        return 0;
    }
    // K cut in pieces: 32-bit partial sums [piece][M][N] in the workspace, added in order by the
    // caller's next kernel or by the reduce kernel here
    int k_per_split = round_up(ceil_div(k, splits), 128 / (int)sizeof(E));
    splits = ceil_div(k, k_per_split);
    gemm_mfma_kernel<EPI_F32, T, E><<<round_up(n_tiles * splits, 8), T::THREADS, T::LDS_BYTES, stream>>>(
        (const E*)x, ldx, (const E*)w, ldw, workspace, n, m, n, k, tiles_m, n_tiles, k_per_split,
        (long long)m * n);
    if (plan.defer && ldo == n) {
        *plan.deferred = splits;
        return 0;
    }
    long long total = (long long)m * n;
    gemm_splitk_reduce_kernel<EPI><<<ceil_div(total, 256), 256, 0, stream>>>((const float*)workspace, out, ldo, m, n, splits);
    return 0;
}

// The ring kernel.
template <int EPI, typename T, typename E = bf16_t>
static int launch_ring(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m,
                       int n, int k, int splits, void* workspace, SplitPlan plan, hipStream_t stream) {
    static bool ready = false;
    if (!ready) {
        if (allow_lds(gemm_ring_kernel<EPI, T, E>, T::LDS_BYTES, "gemm")) return 1;
        if (allow_lds(gemm_ring_kernel<EPI_F32, T, E>, T::LDS_BYTES, "gemm")) return 1;
        ready = true;
    }
    int tiles_m = ceil_div(m, T::BM), tiles_n = ceil_div(n, T::BN);
    int n_tiles = tiles_m * tiles_n;
    if (splits <= 1) {
        gemm_ring_kernel<EPI, T, E><<<round_up(n_tiles, 8), T::THREADS, T::LDS_BYTES, stream>>>(
            (const E*)x, ldx, (const E*)w, ldw, out, ldo, m, n, k, tiles_m, n_tiles, k, 0);
        return 0;
    }
    int k_per_split = round_up(ceil_div(k, splits), 128 / (int)sizeof(E));
    splits = ceil_div(k, k_per_split);
    gemm_ring_kernel<EPI_F32, T, E><<<round_up(n_tiles * splits, 8), T::THREADS, T::LDS_BYTES, stream>>>(
        (const E*)x, ldx, (const E*)w, ldw, workspace, n, m, n, k, tiles_m, n_tiles, k_per_split,
        (long long)m * n);
    if (plan.defer && ldo == n) {
        *plan.deferred = splits;
        return 0;
    }
    long long total = (long long)m * n;
    gemm_splitk_reduce_kernel<EPI><<<ceil_div(total, 256), 256, 0, stream>>>((const float*)workspace, out, ldo, m, n, splits);
    return 0;
}

// The same for the 256x256 kernel: one block a CU walks through its share of the tiles (and K pieces).
template <int EPI>
static int launch_pingpong(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m, int n, int k,
                           int splits, void* workspace, SplitPlan plan, hipStream_t stream) {
    static bool ready = false;
    if (!ready) {
        if (allow_lds(gemm_pingpong_kernel<EPI>, pingpong::LDS_BYTES, "gemm")) return 1;
        if (allow_lds(gemm_pingpong_kernel<EPI_F32>, pingpong::LDS_BYTES, "gemm")) return 1;
        ready = true;
    }
    const int tiles_m = ceil_div(m, 256), n_tiles = tiles_m * ceil_div(n, 256);
    int k_per_split = splits <= 1 ? k : round_up(ceil_div(k, splits), GM_BK);
    splits = ceil_div(k, k_per_split);
    const int items = n_tiles * splits, cus = cu_count() / 8 * 8;
    const int blocks = cus > 0 && round_up(items, 8) > cus ? cus : round_up(items, 8);
    if (splits <= 1) {
        gemm_pingpong_kernel<EPI><<<blocks, 512, pingpong::LDS_BYTES, stream>>>(
            (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, out, ldo, m, n, k, tiles_m, n_tiles, k, 0, items);
        return 0;
    }
    gemm_pingpong_kernel<EPI_F32><<<blocks, 512, pingpong::LDS_BYTES, stream>>>(
        (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, workspace, n, m, n, k, tiles_m, n_tiles, k_per_split, (long long)m * n, items);
    if (plan.defer && ldo == n) {
        *plan.deferred = splits;
        return 0;
    }
    gemm_splitk_reduce_kernel<EPI><<<ceil_div((long long)m * n, 256), 256, 0, stream>>>((const float*)workspace, out, ldo, m, n, splits);
    return 0;
}

// The tile shapes of the many-rows kernels, as rows x columns of a block's tile (the number is the algorithm that asks for one):
// 256x256 is gemm_pingpong_kernel's, 256x192 (eight waves of 64x96) gemm_mfma_kernel's, whose LDS stages are too large for a
// ring of three, the others are the ring kernel's.  What one costs: how many blocks a CU holds (`cap`), microseconds per 64-wide
// K stage for a CU that holds as many blocks as fit when half the chip or less is at work (`light`) and when all of it is
// (`full`: the L2s are shared and the clock drops under load), for a CU that holds one of two (`alone`), what a launch costs
// beside its stages (`fixed`) and every further round of blocks (`round`), the rate at which weights arrive (`weights`, TB/s) and
// sums leave (`sums`).
struct TileKind { int bm, bn, cap; double light, full, alone, fixed, round, weights, sums; int algo; };
static const TileKind TILE_KINDS[] = {
    {256, 256, 1, 1.06, 1.38, 0.0, 7.00, 2.05, 7.95, 5.15, ALGO_MFMA_TILE256},     {256, 192, 1, 0.91, 1.28, 0.0, 6.40, 8.90, 7.80, 6.35, ALGO_MFMA_TILE256X192},
    {128, 128, 1, 0.459, 0.529, 0.0, 3.68, 2.15, 5.26, 4.38, ALGO_MFMA_TILE},      {64, 64, 2, 0.474, 0.452, 0.253, 2.60, 0.69, 5.50, 5.08, ALGO_MFMA_TILE64},
    {128, 64, 2, 0.682, 0.677, 0.385, 2.64, 0.77, 4.98, 4.78, ALGO_MFMA_TILE128X64}, {128, 192, 1, 0.617, 0.697, 0.0, 4.56, 3.11, 5.53, 4.91, ALGO_MFMA_TILE128X192},
    {256, 128, 1, 0.665, 0.812, 0.0, 5.64, 4.17, 4.98, 6.29, ALGO_MFMA_TILE256X128}, {128, 256, 1, 0.780, 0.834, 0.0, 4.94, 3.35, 5.70, 5.39, ALGO_MFMA_TILE128X256},
    {64, 128, 1, 0.385, 0.395, 0.0, 3.44, 1.79, 5.89, 4.74, ALGO_MFMA_TILE64X128}};

// An estimate of a product's time in microseconds with tiles of `kind` and K cut into `pieces` (each piece the work of a block of
// its own, 32-bit partial sums written once here and read once by whoever adds them): the rounds of blocks the chip holds at a
// time, each round its K stages at the rate of the CUs' load or at that of the weights that its blocks pull (a strip is read by
// all tile rows at once, from memory once), whichever is slower, both where they are alike; a fixed part for the launch and one
// for every further round; the bytes the epilogue moves.
// The constants are a fit to 34,867 times of 2,719 products (17 to 3,000 rows, 18 outputs from 520 to 34816, K from 256 to 12288;
// left to the next kernel, whole, gated; weights from memory), those within twice the best.  The estimate is 5 to 9 % off (root mean
// square), the choice by it 0.9 % behind the best on average, more than 5 % for 186 products and 28 % at worst.
// Those of the two 256-row kinds were searched for afterwards by the choice's loss, over 77,803 times of 1,874 products (outputs up to
// 151936, every kind, whole and in pieces) and 5,316 of layers' own products at 512 to 16,384 rows (the first fit had 256x256 a fifth too slow).  Microseconds, by the first choice and by this
// one: gated 384 rows x 24576 x 4096 104 -> 90 (256x256 for 128x192), 512 x 32768 x 2048 76 -> 59, 160 x 151936 x 2560 254 -> 221; on
// average 0.5 % behind the best of the gated products (1.0), 1.0 of the whole (1.3) and 1.1 of those left to the next kernel (1.5).
static double tile_cost(const TileKind& kind, int pieces, int m, int n, int k, int epi, bool defer, int cus) {
    const int tiles_m = ceil_div(m, kind.bm);
    const long long tiles = (long long)tiles_m * ceil_div(n, kind.bn);
    const int k_per_piece = round_up(ceil_div(k, pieces), GM_BK);
    pieces = ceil_div(k, k_per_piece);
    const long long blocks = tiles * pieces, slots = (long long)cus * kind.cap;
    const double stages = (double)(k_per_piece / GM_BK);
    auto stage_us = [&](long long together) {          // blocks on the chip at the same time, at most `slots`
        double share = (double)together / (double)cus, busy = (double)together / (double)slots;
        double w = busy <= 0.5 ? 0.0 : busy >= 1.0 ? 1.0 : (busy - 0.5) * 2.0;
        double own = kind.light + (kind.full - kind.light) * w;
        if (kind.cap == 2 && together <= cus) own = kind.alone * (1.0 + 0.2 * (share > 0.5 ? share - 0.5 : 0.0));
        double arrive = (double)together / tiles_m * kind.bn * (GM_BK * 2.0) / (kind.weights * 1e6);
        return cbrt(own * own * own + arrive * arrive * arrive);
    };
    const long long rounds = blocks / slots, rest = blocks % slots;
    double t = (rounds ? (double)rounds * stages * stage_us(slots) : 0.0) + (rest ? stages * stage_us(rest) : 0.0);
    t += kind.fixed + kind.round * (double)(rounds + (rest ? 1 : 0) - 1);
    const double moved = epi_gated(epi) ? (double)m * n : (double)m * n * 4.0 * (pieces > 1 ? pieces : epi == EPI_ACC ? 2.0 : 1.0);
    t += moved / (kind.sums * 1e6);
    if (pieces > 1) t += (double)pieces * m * n * 4.0 / 5.0e6 + (defer ? 0.0 : 3.96);   // read again, by a kernel of their own unless deferred
    return t;
}

// The 256x256 and the ring kernel address a tile's rows by 31-bit offsets.
static bool rows_near(int ldx, int ldw, int size) { return (long long)(ldx > ldw ? ldx : ldw) * 256 * size < 0x7fff0000ll; }

#include "gemm_f32.h"

// algo: ALGO_AUTO = choose, else the tile kernel asked for (then K stays whole).  The choice is the smallest estimate over shapes and
// pieces.  What counts is the CU with the most work and how fast a tile's stage goes: 34816 columns at 192 rows are 136 tiles of
// 256, little more than half of the chip, or 182 of 192 (105 us for 120); 6144 columns at 2,048 rows are 192 tiles of 256 or 256 of 192, whose
// stages on a full chip are slower by more (91 us for 95).  A product with few tiles (few rows, or a narrow output)
// leaves most CUs idle while a few walk through all of K: then K is cut into pieces of at least 256 (512 where more than eight).
struct TileChoice { int algo, pieces; };

static TileChoice choose_tile(int m, int n, int k, int epi, bool defer, bool near, int most, int cus) {
    // (a step asks for the same few products over and over: the last answers are kept)
    struct Kept { int m, n, k, epi, defer, near, most, cus; TileChoice choice; };
    static thread_local Kept kept[64];
    Kept& slot = kept[((unsigned)n * 31u + (unsigned)k * 7u + (unsigned)m) % 64u];
    if (slot.m == m && slot.n == n && slot.k == k && slot.epi == epi && slot.defer == defer && slot.near == near && slot.most == most && slot.cus == cus)
        return slot.choice;
    TileChoice choice{ALGO_MFMA_TILE256X192, 1};
    double best = 1e30;
    // From 256 rows and K of 4096 on, a K with a rest of a stage keeps 256x256 tiles and with them the number of pieces that a
    // caller who adds them up has been given for such sizes (the ring in fewer pieces is 4 to 19 % faster: 402 x 4046 x 9328 73 us
    // in seven, 61 in four); the estimates were fitted to whole stages.
    const bool rest = k % GM_BK != 0 && k >= 4096 && m >= 256;
    for (const auto& kind : TILE_KINDS) {
        if (near ? rest && kind.algo != ALGO_MFMA_TILE256 : kind.algo != ALGO_MFMA_TILE256X192) continue;
        for (int pieces = 1; pieces <= most && (pieces == 1 || k / pieces >= (pieces <= 8 ? 256 : 512)); ++pieces) {
            double t = tile_cost(kind, pieces, m, n, k, epi, defer, cus);
            if (t < best) { best = t; choice = {kind.algo, pieces}; }
        }
    }
    slot = Kept{m, n, k, epi, defer, near, most, cus, choice};
    return choice;
}

// The algorithm whose tiles a bfloat16 product of many rows takes when K stays whole (gated: with the gated activation).
ROCML_EXPORT int rocml_gemm_tile_algo(int m, int n, int k, int gated) {
    if (m < 1 || n < 1 || k < 1) return ALGO_AUTO;
    return choose_tile(m, n, k, gated ? EPI_SWIGLU : EPI_F32, false, true, 1, cu_count()).algo;
}

template <int EPI>
static int launch_mfma_tile(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m,
                            int n, int k, int algo, void* workspace, long long workspace_bytes, SplitPlan plan,
                            hipStream_t stream) {
    const bool near = rows_near(ldx, ldw, 2);
    int splits = 1;
    if (algo == ALGO_AUTO) {
        long long most = epi_gated(EPI) || !workspace ? 1 : workspace_bytes / ((long long)m * n * (long long)sizeof(float));
        most = most > 16 ? 16 : most;
        most = most > plan.max_splits ? plan.max_splits : most;
        TileChoice c = choose_tile(m, n, k, EPI, plan.defer && ldo == n, near, most < 1 ? 1 : (int)most, cu_count());
        algo = c.algo;
        splits = c.pieces;
    }
    if (!near) algo = ALGO_MFMA_TILE256X192;
#define RING(S_, ...) launch_ring<EPI, RingTile<GemmTile<__VA_ARGS__>, S_>>(x, ldx, w, ldw, out, ldo, m, n, k, splits, workspace, plan, stream)
    switch (algo) {
        case ALGO_MFMA_TILE256: return launch_pingpong<EPI>(x, ldx, w, ldw, out, ldo, m, n, k, splits, workspace, plan, stream);
        case ALGO_MFMA_TILE256X192: return launch_mfma_tile_as<EPI, GemmTile192>(x, ldx, w, ldw, out, ldo, m, n, k, splits, workspace, plan, stream);
        case ALGO_MFMA_TILE128X192: return RING(4, 4, 2, 1, 3);
        case ALGO_MFMA_TILE256X128: return RING(3, 4, 2, 2, 2);
        case ALGO_MFMA_TILE64X128: return RING(6, 2, 2, 1, 2);
        case ALGO_MFMA_TILE64: return RING(4, 2, 2, 1, 1);
        case ALGO_MFMA_TILE128X64: return RING(3, 2, 2, 2, 1);
        case ALGO_MFMA_TILE128X256: return RING(3, 2, 4, 2, 2);
        default: return RING(4, 4, 2, 1, 2);
    }
#undef RING
}

// The two-steps-ahead kernel on a product that cannot be cut along K (the gated product), with
// WAVES waves a block, each on 16 columns.
template <int MT, int EPI, int WAVES>
static int launch_ahead_whole(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m, int n,
                              int k, RowScale rs, hipStream_t stream) {
    constexpr int LDS = 2 * MT * 16 * GS_ROW * 16;
    static bool ready = false;
    if (!ready) {
        if (allow_lds(gemm_skinny_ahead_kernel<MT, EPI, false, WAVES>, LDS, "gemm")) return 1;
        ready = true;
    }
    gemm_skinny_ahead_kernel<MT, EPI, false, WAVES><<<dim3(ceil_div(n, 16 * WAVES), 1), 64 * WAVES, LDS, stream>>>(
        (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, out, ldo, m, n, k, round_up(k, GS_KC), rs);
    return 0;
}

// Waves a block for such a product.  A CU pulls weight rows in 64-byte runs at a limited rate (the
// kernel's loads put a row's four pieces into the lanes of one instruction) and a second block on
// a CU stages the activations again, so the blocks should be one round that uses every CU: the
// fewest waves whose blocks the chip holds at once.  Measured at 64 rows: 24576 columns in 44 us
// with six waves (256 blocks; eight waves are 192 blocks and leave a quarter of 256 CUs idle:
// 49 us; five are two rounds: 72), 34816 x 5120 in 79 us with nine (eight: 116), 51200 x 5120 in
// 115 us with sixteen (eight: 124).  ``skip_from..skip_to``: counts whose kernel does not fit its
// registers.  A product wider than one round of the largest blocks gets the count that leaves the
// fewest columns on the busiest CU.
static int ahead_waves(int n, int cus, int skip_from, int skip_to) {
    for (int waves = 2; waves <= 16; ++waves)
        if ((waves < skip_from || waves > skip_to) && ceil_div(n, 16 * waves) <= cus) return waves;
    int best = 16, best_cols = 1 << 30;
    for (int waves = 16; waves >= 2; --waves) {
        if (waves >= skip_from && waves <= skip_to) continue;
        int cols = ceil_div(ceil_div(n, 16 * waves), cus) * 16 * waves;
        if (cols < best_cols) {
            best = waves;
            best_cols = cols;
        }
    }
    return best;
}

// The same kernel on one K range of a product that is cut along K: 32-bit partial sums
// [split][M][N] into the workspace.
template <int MT, int WAVES>
static int launch_ahead_split(const void* x, int ldx, const void* w, int ldw, void* workspace, int m, int n, int k,
                              int splits, int k_per_split, hipStream_t stream) {
    constexpr int LDS = 2 * MT * 16 * GS_ROW * 16;
    static bool ready = false;
    if (!ready) {
        if (allow_lds(gemm_skinny_ahead_kernel<MT, EPI_F32, true, WAVES>, LDS, "gemm")) return 1;
        ready = true;
    }
    gemm_skinny_ahead_kernel<MT, EPI_F32, true, WAVES><<<dim3(ceil_div(n, 16 * WAVES), splits), 64 * WAVES, LDS, stream>>>(
        (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, workspace, n, m, n, k, k_per_split);
    return 0;
}

// Blocks of a product that may be cut along K: waves a block (16 columns each) and K pieces, so
// that the CU with the most work has as little as possible: its weight bytes (rounds of blocks
// times a block's columns times its K range) plus its share of the partial sums, which are
// written once and read once.  6144 x 4096 at 8 rows: 64 blocks of six waves times four pieces are
// one round of 256 equal blocks; 96 blocks of four waves times four pieces leave half the CUs with
// two blocks and half with one.
struct BlockChoice { int waves, splits, k_per_split; };

// An estimate of the busiest CU's time in microseconds.  A wave keeps two steps of weights
// (16 KB) on their way for the two microseconds a trip takes, a CU pulls such rows at up to about
// 45 GB/s however many waves ask (measured: 2.9 us more per 16 columns x 4096 a CU), a block
// stages its rows' activations of its K range through LDS once, LDS holds so many blocks of these
// rows at a time, and the partial sums are written here and read by the next kernel.
static double block_cost(BlockChoice c, int m, int row_tiles, int n, int cus) {
    const double lds_block = 2.0 * row_tiles * 16 * GS_ROW * 16;
    const int resident = (int)(160.0 * 1024 / lds_block) < 1 ? 1 : (int)(160.0 * 1024 / lds_block);
    long long blocks = (long long)ceil_div(n, 16 * c.waves) * c.splits;
    int per_cu = (int)ceil_div(blocks, (long long)cus);
    int together = per_cu < resident ? per_cu : resident;
    double rounds = (double)ceil_div(per_cu, together);
    double rate = 8.0e3 * c.waves * together;                              // bytes per microsecond
    if (rate > 45.0e3) rate = 45.0e3;
    double weights = 16.0 * c.waves * c.k_per_split * 2.0 * together;      // of the blocks that run together
    double staged = 16.0 * row_tiles * c.k_per_split * 2.0 * together;
    double cost = rounds * (weights / rate + staged / 100.0e3 + 3.0);
    if (c.splits > 1) cost += (double)c.splits * (m * (double)n * 8.0 / 2.0e6 + 0.15);
    return cost;
}

static BlockChoice choose_blocks(BlockChoice usual, int m, int row_tiles, int n, int k, int cus,
                                 long long workspace_bytes, int skip_from, int skip_to, int max_splits) {
    // (a step asks for the same few products over and over: the last answers are kept)
    // (the answer depends on the usual blocks and on the skipped wave counts too, which differ
    // between the callers that share this table)
    struct Kept { int m, row_tiles, n, k, cus; long long workspace_bytes; BlockChoice usual; int skip_from, skip_to, max_splits;
                  BlockChoice choice; bool set; };
    static thread_local Kept kept[64];
    Kept& slot = kept[((unsigned)n * 31u + (unsigned)k * 7u + (unsigned)m) % 64u];
    if (slot.set && slot.m == m && slot.row_tiles == row_tiles && slot.n == n && slot.k == k && slot.cus == cus &&
        slot.workspace_bytes == workspace_bytes && slot.usual.waves == usual.waves && slot.usual.splits == usual.splits &&
        slot.usual.k_per_split == usual.k_per_split && slot.skip_from == skip_from && slot.skip_to == skip_to &&
        slot.max_splits == max_splits)
        return slot.choice;
    BlockChoice best = usual;
    double best_cost = 1e30;
    for (int kps = GS_KC; kps < k + GS_KC; kps += GS_KC) {
        int splits = ceil_div(k, kps);
        if (splits > max_splits) continue;
        if (splits > 1 && (kps < 2 * GS_KC || (long long)splits * m * n * (long long)sizeof(float) > workspace_bytes)) continue;
        for (int waves = 2; waves <= 16; ++waves) {
            if (waves >= skip_from && waves <= skip_to) continue;
            BlockChoice c{waves, splits, kps};
            double cost = block_cost(c, m, row_tiles, n, cus);
            if (cost < best_cost * 0.999) {
                best_cost = cost;
                best = c;
            }
        }
    }
    // the usual blocks (four or eight waves, about two blocks or one a CU) unless the estimate
    // promises a clear gain: it is rough, and they are what the kernels were tuned with
    BlockChoice choice = best_cost < 0.93 * block_cost(usual, m, row_tiles, n, cus) ? best : usual;
    slot = Kept{m, row_tiles, n, k, cus, workspace_bytes, usual, skip_from, skip_to, max_splits, choice, true};
    return choice;
}

template <int MT, int EPI>
static int launch_skinny(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m, int n,
                         int k, void* workspace, long long workspace_bytes, SplitPlan plan, hipStream_t stream) {
    const int cus = cu_count();
    if constexpr (epi_gated(EPI)) {
        // The gated epilogue needs whole sums: the kernel that requests two steps ahead, whatever
        // the number of rows, with the number of waves that makes its blocks one round.  (At 49 to
        // 64 rows the kernels of 13 to 15 waves need more registers than 832 to 960 threads
        // leave each.)
        switch (ahead_waves(n, cus, MT == 4 ? 13 : 17, MT == 4 ? 15 : 17)) {
#define AHEAD_CASE(W_) case W_: return launch_ahead_whole<MT, EPI, W_>(x, ldx, w, ldw, out, ldo, m, n, k, plan.rs, stream);
            AHEAD_CASE(2) AHEAD_CASE(3) AHEAD_CASE(4) AHEAD_CASE(5) AHEAD_CASE(6) AHEAD_CASE(7) AHEAD_CASE(8)
            AHEAD_CASE(9) AHEAD_CASE(10) AHEAD_CASE(11) AHEAD_CASE(12) AHEAD_CASE(13) AHEAD_CASE(14)
            AHEAD_CASE(15) AHEAD_CASE(16)
#undef AHEAD_CASE
            default: return rocml_fail("gemm: no kernel of that many waves");
        }
    } else {
    constexpr int LDS = 2 * MT * 16 * GS_ROW * 16;
    // Up to 16 rows: four waves per block, or two for the wide products that cannot be split
    // (more, smaller blocks keep more loads in flight when nothing else multiplies their
    // number), about 512 blocks.  Beyond 16 rows the kernel that requests two steps ahead, with
    // eight waves per block (LDS for the activations limits a CU to two blocks at 64 rows;
    // eight waves double the weight bytes in flight per CU and halve the times the activations
    // are read), about 256 blocks.
    constexpr bool AHEAD = MT > 1;
    constexpr int WIDE = AHEAD ? 8 : 4;
    static bool ready = false;
    if (!ready) {
        if constexpr (AHEAD) {
            if (allow_lds(gemm_skinny_ahead_kernel<MT, EPI, false, WIDE>, LDS, "gemm")) return 1;
            if (allow_lds(gemm_skinny_ahead_kernel<MT, EPI, true, WIDE>, LDS, "gemm")) return 1;
        } else {
            if (allow_lds(gemm_skinny_kernel<MT, EPI, false, WIDE>, LDS, "gemm")) return 1;
            if (allow_lds(gemm_skinny_kernel<MT, EPI, true, WIDE>, LDS, "gemm")) return 1;
        }
        ready = true;
    }
    // ("wide" is a product whose blocks of four waves alone are four to a CU or more)
    bool narrow = MT == 1 && n >= 256 * cus;
    int blocks_n = ceil_div(n, narrow ? 32 : 16 * WIDE);
    int target = AHEAD ? cus : 2 * cus;
    int splits = target / blocks_n;
    int by_k = k / 512;
    if (splits > by_k) splits = by_k;
    if (splits > plan.max_splits) splits = plan.max_splits;
    if (splits < 1 || narrow) splits = 1;
    long long per_split = (long long)m * n * sizeof(float);
    if (splits > 1 && (long long)splits * per_split > workspace_bytes)
        splits = workspace ? (int)(workspace_bytes / per_split) : 1;
    if (splits < 1) splits = 1;
    int k_per_split = round_up(ceil_div(k, splits), GS_KC);
    splits = ceil_div(k, k_per_split);
    dim3 grid(blocks_n, splits);
    if (!narrow && workspace) {
        BlockChoice usual{WIDE, splits, k_per_split};
        BlockChoice c = choose_blocks(usual, m, MT, n, k, cus, workspace_bytes, MT == 4 ? 13 : 17, MT == 4 ? 15 : 17, plan.max_splits);
        if (c.splits > 1 && (c.waves != usual.waves || c.splits != usual.splits)) {
            int rc = 1;
            switch (c.waves) {
#define AHEAD_CASE(W_) case W_: rc = launch_ahead_split<MT, W_>(x, ldx, w, ldw, workspace, m, n, k, c.splits, c.k_per_split, stream); break;
                AHEAD_CASE(2) AHEAD_CASE(3) AHEAD_CASE(4) AHEAD_CASE(5) AHEAD_CASE(6) AHEAD_CASE(7) AHEAD_CASE(8)
                AHEAD_CASE(9) AHEAD_CASE(10) AHEAD_CASE(11) AHEAD_CASE(12) AHEAD_CASE(13) AHEAD_CASE(14)
                AHEAD_CASE(15) AHEAD_CASE(16)
#undef AHEAD_CASE
                default: return rocml_fail("gemm: no kernel of that many waves");
            }
            if (rc) return rc;
            if (plan.defer && ldo == n) {
                *plan.deferred = c.splits;
                return 0;
            }
            long long total = (long long)m * n;
            gemm_splitk_reduce_kernel<EPI><<<ceil_div(total, 256), 256, 0, stream>>>(
                (const float*)workspace, out, ldo, m, n, c.splits);
            return 0;
        }
    }
    if (splits == 1 && narrow) {
        if constexpr (MT == 1)
            gemm_skinny_kernel<MT, EPI, false, 2><<<grid, 128, LDS, stream>>>(
                (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, out, ldo, m, n, k, k_per_split);
    } else if (splits == 1) {
        if constexpr (AHEAD)
            gemm_skinny_ahead_kernel<MT, EPI, false, WIDE><<<grid, 64 * WIDE, LDS, stream>>>(
                (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, out, ldo, m, n, k, k_per_split);
        else
            gemm_skinny_kernel<MT, EPI, false, WIDE><<<grid, 64 * WIDE, LDS, stream>>>(
                (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, out, ldo, m, n, k, k_per_split);
    } else {
        if constexpr (AHEAD)
            gemm_skinny_ahead_kernel<MT, EPI, true, WIDE><<<grid, 64 * WIDE, LDS, stream>>>(
                (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, workspace, n, m, n, k, k_per_split);
        else
            gemm_skinny_kernel<MT, EPI, true, WIDE><<<grid, 64 * WIDE, LDS, stream>>>(
                (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, workspace, n, m, n, k, k_per_split);
        if (plan.defer && ldo == n) {
            // the caller's next kernel adds the partial sums itself
            *plan.deferred = splits;
            return 0;
        }
        long long total = (long long)m * n;
        gemm_splitk_reduce_kernel<EPI><<<ceil_div(total, 256), 256, 0, stream>>>(
            (const float*)workspace, out, ldo, m, n, splits);
    }
    return 0;
    }
}

// At most 16 rows: blocks of 16 weight rows, K split over the block's waves and, while there are
// fewer than three blocks a CU, over blocks as well (in pieces of at most 1024: up to 256 of K a wave).
template <int EPI>
static int launch_kpar(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m, int n, int k,
                       void* workspace, long long workspace_bytes, SplitPlan plan, hipStream_t stream) {
    int n_tiles = ceil_div(n, 16);
    // A CU holds three blocks, and four blocks of which the last waits cost more than they bring, but for K below 2048, where a
    // wave has less than a chunk (microseconds at one row, four and three blocks a CU: 8192 x 9728 36.2 and 33.1, 8192 x 3072
    // 14.6 and 12.4, 7168 x 6144 22.2 and 20.8; 8192 x 1536 8.2 and 8.9).
    int splits = (k < 2048 ? 4 : 3) * cu_count() / n_tiles;
    int by_k = ceil_div(k, 1024);                      // (a wave then has one chunk of 256)
    if (splits > by_k) splits = by_k;
    if (splits > plan.max_splits) splits = plan.max_splits;
    // Whole sums spare the reduce kernel: up to K of 2048, and up to 4096 while the blocks are at most one a CU and enough to pull
    // the weights by themselves (microseconds at one row and K of 4096, in pieces and whole: 1024 columns 6.2 and 7.4, 1536 7.3
    // and 7.4, 2048 7.7 and 7.4, 4096 11.9 and 9.4; the few-rows kernel 7.6, 7.7, 8.2 and 10.7).
    const bool deferred = plan.defer && ldo == n;
    if (splits < 1 || epi_gated(EPI) || (!deferred && (k <= 2048 || (k <= 4096 && 8 * n_tiles > 3 * cu_count() && n_tiles <= cu_count())))) splits = 1;
    long long per_split = (long long)m * n * sizeof(float);
    if (splits > 1 && (long long)splits * per_split > workspace_bytes)
        splits = workspace ? (int)(workspace_bytes / per_split) : 1;
    if (splits < 1) splits = 1;
    int k_per_split = round_up(ceil_div(k, splits), 128);
    splits = ceil_div(k, k_per_split);
    dim3 grid(n_tiles, splits);
    const bool far = ldx >= NEAR_STRIDE || ldw >= NEAR_STRIDE;
#define KPAR(PARTIAL_, FAR_, ...) \
    gemm_kpar_kernel<EPI, PARTIAL_, FAR_><<<grid, GK_THREADS, 0, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)w, ldw, __VA_ARGS__)
    if (splits == 1) {
        if (far) KPAR(false, true, out, ldo, m, n, k, k_per_split, plan.rs);
        else KPAR(false, false, out, ldo, m, n, k, k_per_split, plan.rs);
    } else {
        if (far) KPAR(true, true, workspace, n, m, n, k, k_per_split, RowScale{});
        else KPAR(true, false, workspace, n, m, n, k, k_per_split, RowScale{});
#undef KPAR
        if (plan.defer && ldo == n) {
            *plan.deferred = splits;
            return 0;
        }
        long long total = (long long)m * n;
        gemm_splitk_reduce_kernel<EPI><<<ceil_div(total, 256), 256, 0, stream>>>(
            (const float*)workspace, out, ldo, m, n, splits);
    }
    return 0;
}

template <int EPI>
static int launch_skinny_m(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int m, int n,
                           int k, void* workspace, long long workspace_bytes, SplitPlan plan, hipStream_t stream) {
    if (m <= 16) return launch_skinny<1, EPI>(x, ldx, w, ldw, out, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
    if (m <= 32) return launch_skinny<2, EPI>(x, ldx, w, ldw, out, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
    if (m <= 48) return launch_skinny<3, EPI>(x, ldx, w, ldw, out, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
    return launch_skinny<4, EPI>(x, ldx, w, ldw, out, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
}

// Gated activation over a 32-bit [M, N] product with (gate, up) column pairs: the unfused path of
// the epilogue above, for the kernels that cannot fuse it.
template <typename TO>
__global__ void swiglu_pairs_kernel(const float* __restrict__ gu, TO* __restrict__ out, int ldo, int m, int half, int relu) {
    long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)m * half) return;
    int r = (int)(idx / half), j = (int)(idx - (long long)r * half);
    const float* row = gu + (size_t)r * 2 * half;
    Elem<TO>::store(out + (size_t)r * ldo + j, relu ? fmaxf(row[2 * j], 0.f) * row[2 * j + 1] : silu_mul(row[2 * j], row[2 * j + 1]));
}

// out (+)= sum of split-K partial sums [splits][M][N] in split order: the step that a deferred
// product leaves to its caller, as a kernel of its own.
ROCML_EXPORT int rocml_splitk_reduce(const float* partials, void* out, int out_dtype, int ldo, int m, int n,
                                     int splits, int accumulate, hipStream_t stream) {
    ROCML_REQUIRE(m >= 0 && n > 0 && splits > 0 && ldo >= n, "splitk_reduce: bad sizes M=%d N=%d splits=%d", m, n, splits);
    ROCML_REQUIRE(!accumulate || out_dtype == ROCML_F32, "splitk_reduce: accumulation needs a 32-bit output");
    if (m == 0) return 0;
    int grid = ceil_div((long long)m * n, 256);
    if (accumulate) gemm_splitk_reduce_kernel<EPI_ACC><<<grid, 256, 0, stream>>>(partials, out, ldo, m, n, splits);
    else if (out_dtype == ROCML_F32) gemm_splitk_reduce_kernel<EPI_F32><<<grid, 256, 0, stream>>>(partials, out, ldo, m, n, splits);
    else if (out_dtype == ROCML_BF16) gemm_splitk_reduce_kernel<EPI_BF16><<<grid, 256, 0, stream>>>(partials, out, ldo, m, n, splits);
    else return rocml_fail("splitk_reduce: unknown output type %d", out_dtype);
    ROCML_CHECK_LAUNCH("splitk_reduce");
    return 0;
}

// Waves of a block of the kernel below: few enough that a wave's share of K is one chunk of 256, for one trip to memory
// (microseconds at one row: 1024 x 2048 5.8 with four waves, 4.8 with eight; 1024 x 3072 7.6, 6.8 and 6.1 with twelve);
// beyond 3072 the count of eight or twelve with fewer chunks (4096 x 12288: 21.5 and 21.0; 2048 x 6144: 10.3 and 10.0).
static int prescale_waves(int k) {
    if (k <= 3072) return k <= 1024 ? 4 : k <= 2048 ? 8 : 12;
    return ceil_div(ceil_div(k, 12), 256) < ceil_div(ceil_div(k, 8), 256) ? 12 : 8;
}

// resid[M, N] += X * W^T for at most 16 rows of bfloat16 operands, whole sums, and the next norm
// prepared: xg[M, N] = bfloat16(resid * gain) and ssq[M][ceil(N / 16)], the sums of squares of
// every 16 columns of a row (see gemm_residual_prescale_kernel).
ROCML_EXPORT int rocml_gemm_residual_prescale(const void* x, int ldx, const void* w, int ldw, float* resid, int ldr,
                                              const float* gain, void* xg, int ldg, float* ssq, int m, int n, int k,
                                              int waves, const float* bias, hipStream_t stream) {
    ROCML_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm_residual_prescale: bad sizes M=%d N=%d K=%d", m, n, k);
    ROCML_REQUIRE(m <= 16, "gemm_residual_prescale: at most 16 rows, got %d", m);
    ROCML_REQUIRE(ldx >= k && ldw >= k && ldr >= n && ldg >= n, "gemm_residual_prescale: row strides (%d, %d, %d, %d) too small",
                  ldx, ldw, ldr, ldg);
    ROCML_REQUIRE(k % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0,
                  "gemm_residual_prescale: K and the operands' row strides must be multiples of 8 and the pointers "
                  "16-byte aligned (K=%d ldx=%d ldw=%d)", k, ldx, ldw);
    ROCML_REQUIRE((uintptr_t)resid % 16 == 0 && (uintptr_t)gain % 16 == 0 && (uintptr_t)xg % 8 == 0 && (uintptr_t)bias % 16 == 0,
                  "gemm_residual_prescale: the residual stream, the gain, the bias and the prepared operand must be aligned");
    ROCML_REQUIRE(resid && gain && xg && ssq, "gemm_residual_prescale: null pointer");
    if (m == 0) return 0;
    int tiles = ceil_div(n, 16);
    ROCML_REQUIRE(waves == 0 || waves == 4 || waves == 8 || waves == 12 || waves == 16,
                  "gemm_residual_prescale: 4, 8, 12 or 16 waves, got %d", waves);
    if (waves == 0) waves = prescale_waves(k);       // (16 only for a caller that asks: 8.8 us for 8.4 with eight at K of 4096)
    const bool one = round_up(ceil_div(k, waves), 32) <= 256;
#define GRP_LAUNCH(W_, ...)                                                                                     \
    gemm_residual_prescale_kernel<W_, __VA_ARGS__><<<tiles, 64 * W_, 0, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)w, ldw, resid, \
                                                                     ldr, gain, (bf16_t*)xg, ldg, ssq, tiles, m, n, k, bias)
    if (ldx >= NEAR_STRIDE || ldw >= NEAR_STRIDE) GRP_LAUNCH(4, false, true);
    else if (waves == 16) { if (one) GRP_LAUNCH(16, true); else GRP_LAUNCH(16, false); }
    else if (waves == 12) { if (one) GRP_LAUNCH(12, true); else GRP_LAUNCH(12, false); }
    else if (waves == 8) { if (one) GRP_LAUNCH(8, true); else GRP_LAUNCH(8, false); }
    else { if (one) GRP_LAUNCH(4, true); else GRP_LAUNCH(4, false); }
#undef GRP_LAUNCH
    ROCML_CHECK_LAUNCH("gemm_residual_prescale");
    return 0;
}

// Whether rocml_gemm_residual_prescale is the faster way to add this product to the residual
// stream and norm the result.  Its blocks own 16 columns and all of K, so the chip must hold them in
// one round, and a CU pulls a block's weight rows at a limited rate, so K must be short or the
// blocks must be nearly one a CU.  Measured in replayed graphs against the product cut along K over
// blocks (the norm kernel behind it takes 4.4 more; us): 4096 x 4096 8.4 against 8.1 at 1 row, 9.5 against 8.4 at
// 8, 10.9 against 9.0 at 16; 1024 x 3072 6.1 against 5.6 at 1 row, 8.2 against 5.9 at 16; 2048 x 6144 10.0 against 7.8 at
// 1 row, 11.1 against 7.6 at 4, 12.1 against 7.7 at 8; 4096 x 12288 21.5 against 20.6 at 1 row, 24.0 against 20.9 at 8 (every
// block reads all activations, which is what more rows cost); 2560 x 9728 (160 blocks) 15.9 against
// 11.6 at 1 row and 5120 x 5120 (320 blocks, more than a round): not taken.  Between K of 4096 and 8192, up to 4 rows: as far as
// a wave of twelve has two chunks (K of 6144) it is ahead of product and norm by 0.9 to 1.8 us at 2048 columns and 1.1 to 3.1
// at 2560; a third chunk costs 0.8 to 1.5 us more than it saves at 2048 and up to 0.9 at 2560, and is 0.5 to 2.3 ahead at 3072.
ROCML_EXPORT int rocml_gemm_residual_prescale_pays(int m, int n, int k) {
    if (m < 1 || m > 16 || k % 8 != 0) return 0;
    int tiles = ceil_div(n, 16);
    const int cus = cu_count();
    if (tiles > cus) return 0;
    if (k <= 4096) return 1;
    if (k <= 8192 && m <= 4 && (k <= 6144 ? 2 : 4) * tiles >= (k <= 6144 ? 1 : 3) * cus) return 1;
    return k <= 12288 && m <= 8 && 10 * tiles >= 9 * cus;
}

// Whether the kernel whose waves split K is the faster one for up to 16 rows where K in pieces of 1024 leaves a wave one chunk of
// 256 and the next kernel adds the pieces: one trip to memory without staging and with half the partial sums of the few-rows
// kernel.  Compared with that kernel on 6,594 products of 1 to 16 rows (15 outputs from 520 to 24576, K from 256 to 12288):
//  * at most one block a CU: 10 to 25 % faster (4096 x 1024 5.0 us for 5.5 at one row, 2048 x 2048 4.4 for 5.4), but whole sums of
//    640 to 896, which the few-rows kernel cuts in two small pieces, 2 to 20 % slower (2048 x 768 1.02 to 1.08 times at 3 to 16 rows);
//  * more than one: the CUs with a block more than the others decide.  A chunk that is half full is still ahead (K of 512: 5 to
//    12 %; of 256, where staging costs nothing, 12 % behind), two pieces where the second round is nearly whole (4096 x 1536 0.92
//    times, 2560 x 1408 1.09 to 1.19), more pieces than two equal, with half the pieces for the next kernel; whole sums
//    of 1024 are 6 to 20 % behind (5120 x 1024 6.2 us for 5.5 at one row, 7.2 for 6.0 at 16).
// From 48 K outputs on the few-rows kernel leaves a K of up to 768 whole, and is 12 to 33 % behind.
static bool kpar_pieces_pay(int m, int n, int k, int cus) {
    const int pieces = ceil_div(k, 1024), blocks = ceil_div(n, 16) * pieces;
    if (k > 512 && k <= 768 && (long long)m * n >= 48 * 1024) return true;
    if (blocks <= cus) return pieces > 1 || k <= 512 || k > 960;
    return k > 2048 || (k > 256 && k <= 512) || (pieces == 2 && 8 * blocks >= 14 * cus && ceil_div(k, 2) <= 960);
}

// The same for sums that must be whole (the gated product, or pieces that nobody would add), up to 8 rows.  K of up to 2048 (gated,
// microseconds at 1 and 8 rows against the few-rows kernel: 12288 x 2048 11.5 and 13.0 for 14.0 and 13.7, 8192 x 2048 8.7 and 10.1
// for 11.9 and 11.8, 6144 x 1024 5.3 and 6.0 for 6.0 and 6.0), and up to two rows K of 4096 in whole chunks (24576 x 4096 38.0 for
// 39.1 at one row, 41.5 for 36.4 at 8).  With more than one block a CU the last chunk of a wave must be worth its trip, the more
// so the more rows there are (times of the few-rows kernel's, 5120 columns: K of 1280 1.06 at 1 row, 1.10 at 4 and 1.17 at 8, 1536 0.98,
// 1.06 and 1.12, 1792 0.88, 0.97 and 1.02; K of 256 1.03 to 1.16).  A product whose pieces nobody adds pays a kernel for them in the
// few-rows kernel: there only K of 256 is behind (1.05 to 1.24), and K beyond 2048 is taken for at most one block a CU
// (5000 x 4096 at one row: 13.1 whole, 16.1 in pieces, 12.5 in the few-rows kernel).
static bool kpar_whole_pays(int m, int n, int k, bool gated, int cus) {
    const bool narrow = n <= 16 * cus;                // at most one block a CU
    if (m <= 2 && k <= 4096 && k % 1024 == 0 && (gated || narrow)) return true;
    if (m > 8 || k > 2048 || n > 48 * cus) return false;
    if (narrow) return true;
    const int last = (k - 1) % 1024 + 1, least = 128 * (m <= 2 ? 2 : m);
    return gated ? last > (least < 768 ? least : 768) : k > 256;
}

// algo: 0 = choose, 1 = plain tiled kernel, 2 = MFMA tile kernel (128x128 tiles), 3 = MFMA few-rows
// kernel (M <= 64), 4 = MFMA kernel for at most 16 rows, 5 to 12 = MFMA tile kernels with 256x256, 256x192, 128x192,
// 256x128, 64x128, 64x64, 128x64 and 128x256 tiles.
// accumulate: out += product (out must be 32-bit); this is the residual sum's epilogue.
// epilogue: 0 = none; 1 = gated activation: W's rows are (gate_j, up_j) pairs and out is
//   [M, N/2] = silu(gate) * up; 2 = the same with max(gate, 0) * up; 3 = max(sum, 0)^2, bfloat16.
// defer: if the product was split along K, leave the partial sums [splits][M][N] at the start of
//   the workspace and report their number in *deferred_splits (0 if the product is complete);
//   the caller's next kernel adds them.  Needs a dense out (ldo == N).
// workspace: device memory for split-K partial sums (may be null: no split).
// row_ssq (may be null): X is bfloat16(x * gain) of a norm over K values whose scale is still to
//   come: row_ssq[M][row_parts] are sums of squares of x whose total over a row gives the row's
//   scale 1 / sqrt(total / K + row_eps), which the gated epilogue applies to its sums.  Only for
//   the gated epilogue of at most 16 rows on the MFMA path.
// max_splits: the most pieces K may be cut into (0: the kernels' own limit of 16), for a caller
//   whose next kernel adds a few partial sums cheaply and more of them one after the other.
ROCML_EXPORT int rocml_gemm(const void* x, int x_dtype, int ldx, const void* w, int w_dtype, int ldw,
                            void* out, int out_dtype, int ldo, int m, int n, int k, int accumulate,
                            int algo, int epilogue, int defer, int* deferred_splits, void* workspace,
                            long long workspace_bytes, const float* row_ssq, int row_parts, float row_eps,
                            int max_splits, hipStream_t stream) {
    if (deferred_splits) *deferred_splits = 0;
    ROCML_REQUIRE(m >= 0 && n > 0 && k > 0, "gemm: bad sizes M=%d N=%d K=%d", m, n, k);
    bool gated = epilogue == 1 || epilogue == 2;        // 1: silu(gate) * up, 2: max(gate, 0) * up
    bool relu2 = epilogue == 3;                         // max(sum, 0)^2
    ROCML_REQUIRE(epilogue >= 0 && epilogue <= 3, "gemm: unknown epilogue %d", epilogue);
    ROCML_REQUIRE(!relu2 || (!accumulate && !defer && x_dtype == ROCML_BF16 && out_dtype == ROCML_BF16),
                  "gemm: the squared-rectifier epilogue stores whole sums of bfloat16 operands as bfloat16");
    ROCML_REQUIRE(!gated || (n % 2 == 0 && !accumulate), "gemm: the gated epilogue needs an even N and no accumulation");
    int out_cols = gated ? n / 2 : n;
    ROCML_REQUIRE(ldx >= k && ldw >= k && ldo >= out_cols, "gemm: row strides (%d, %d, %d) below (K, K, N)",
                  ldx, ldw, ldo);
    ROCML_REQUIRE(!accumulate || out_dtype == ROCML_F32, "gemm: accumulation needs a 32-bit output");
    ROCML_REQUIRE(algo >= ALGO_AUTO && algo <= ALGO_MFMA_TILE128X256, "gemm: unknown algorithm %d", algo);
    ROCML_REQUIRE(!defer || deferred_splits, "gemm: deferring needs a place to report the splits");
    if (m == 0) return 0;
    bool bf16_in = x_dtype == ROCML_BF16 && w_dtype == ROCML_BF16;
    bool mfma_ok = bf16_in && k % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 &&
                   ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0) && (!gated || out_dtype == ROCML_BF16);
    if (algo >= ALGO_MFMA_TILE)
        ROCML_REQUIRE(mfma_ok, "gemm: the MFMA kernels need bfloat16 operands, K and row strides that are "
                               "multiples of 8 and 16-byte aligned pointers (K=%d ldx=%d ldw=%d)", k, ldx, ldw);
    if (algo == ALGO_MFMA_SKINNY)
        ROCML_REQUIRE(m <= 64, "gemm: the few-rows kernel takes at most 64 rows, got %d", m);
    if (algo == ALGO_MFMA_KPAR)
        ROCML_REQUIRE(m <= 16, "gemm: the 16-rows kernel takes at most 16 rows, got %d", m);
    ROCML_REQUIRE(out_dtype == ROCML_F32 || out_dtype == ROCML_BF16, "gemm: unknown output type %d", out_dtype);
    int epi = relu2 ? EPI_RELU2 : gated ? (epilogue == 2 ? EPI_RELUGLU : EPI_SWIGLU) : accumulate ? EPI_ACC : (out_dtype == ROCML_BF16 ? EPI_BF16 : EPI_F32);
    bool use_mfma = mfma_ok && algo != ALGO_PLAIN;
    if (row_ssq)
        ROCML_REQUIRE(gated && m <= 16 && use_mfma && row_parts > 0 && row_eps > 0.f &&
                          (algo == ALGO_AUTO || algo == ALGO_MFMA_SKINNY || algo == ALGO_MFMA_KPAR),
                      "gemm: a row scale goes with the gated epilogue of at most 16 rows on the few-rows MFMA kernels "
                      "(M=%d parts=%d)", m, row_parts);
    if (use_mfma) {
        // Up to 16 rows the few-rows kernels.  Beyond them the ring kernel's pieces of K are ahead of theirs (17 to 48 rows, 1,400 products
        // left to the next kernel or not: 0.5 to 0.9 times their time) but for weights of some 110 MB and more up to 32 rows and 300 MB up
        // to 48, whose blocks a CU are many either way (7168 x 8192 at 23 rows 27 us for 32, 19456 x 12288 at 35 99 for 119; 9728 x
        // 8192 at 20 equal).  The gated product cannot be cut along K: up to 32 rows, and 48 where K is longer than twelve
        // stages of the ring, the few-rows kernel (4 to 9 % ahead; behind by 16 % for K of up to 768 at 33 to 48 rows), and up to 64 for
        // weights of 80 MB and more (19456 x 2560 at 64 27 us for 31, 34816 x 5120 74 for 76; 12288 x 2048 18 for 15).
        const int cus = cu_count();
        const long long weights = (long long)n * k;
        bool few_rows = m <= 16 || (gated ? m <= 32 || (m <= 48 && k > 768) || (m <= 64 && weights >= 40000000)
                                          : n < 256 * cus && weights >= (m <= 32 ? 56000000 : 150000000) && m <= 48);
        bool skinny = algo == ALGO_MFMA_SKINNY || (algo == ALGO_AUTO && few_rows);
        SplitPlan plan{defer, deferred_splits, RowScale{row_ssq, row_parts, row_eps, 1.0f / (float)k},
                       max_splits >= 1 && max_splits < 16 ? max_splits : 16};
        int rc;
#define BY_EPI(fn, ...)                                              \
        (epi == EPI_F32 ? fn<EPI_F32>(__VA_ARGS__)                   \
         : epi == EPI_BF16 ? fn<EPI_BF16>(__VA_ARGS__)               \
         : epi == EPI_ACC ? fn<EPI_ACC>(__VA_ARGS__)                 \
         : epi == EPI_RELU2 ? fn<EPI_RELU2>(__VA_ARGS__)             \
         : epi == EPI_RELUGLU ? fn<EPI_RELUGLU>(__VA_ARGS__) : fn<EPI_SWIGLU>(__VA_ARGS__))
        // The kernel whose waves split K: where K in pieces of 1024 leaves a wave one chunk, where sums must be whole, and
        // for one or two rows against a wide output (at least one and a half blocks of 16 weight rows a CU; beyond two
        // rows the activations read from L2 cost more than the block sharing of the few-rows kernel).
        const long long pieces = ceil_div(k, 1024), kpar_blocks = ceil_div(n, 16) * pieces;
        const bool deferred = plan.defer && ldo == n;
        bool one_trip = m <= 16 && !gated && (pieces == 1 || (workspace && deferred)) && pieces <= plan.max_splits &&
                        2 * kpar_blocks <= (m <= 8 ? 4 : 3) * (long long)cus && pieces * m * n * 4 <= workspace_bytes + (pieces == 1 ? (1ll << 60) : 0) &&
                        (deferred ? kpar_pieces_pay(m, n, k, cus) : k > 256 || n <= 16 * cus);
        bool whole = (gated || !deferred) && kpar_whole_pays(m, n, k, gated, cus);
        bool kpar = algo == ALGO_MFMA_KPAR || (algo == ALGO_AUTO && (one_trip || whole || (m <= 2 && !gated && 2 * (n / 16) >= 3 * cus)));
        if (kpar) rc = BY_EPI(launch_kpar, x, ldx, w, ldw, out, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
        else if (skinny) rc = BY_EPI(launch_skinny_m, x, ldx, w, ldw, out, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
        else rc = BY_EPI(launch_mfma_tile, x, ldx, w, ldw, out, ldo, m, n, k, algo, workspace, workspace_bytes, plan, stream);
#undef BY_EPI
        if (rc) return rc;
        ROCML_CHECK_LAUNCH("gemm");
        return 0;
    }
    // 32-bit operands in 16-byte pieces: the 32-bit matrix instructions, the few-rows kernel while its reads of the
    // activations (every block reads them all) stay below the weights'.  Kernel, tiles and K pieces follow from the number of
    // rows, so a row's sums are rounded in another order in another batch (by about 1e-6 of the row's largest sum); ALGO_PLAIN
    // gives the same bits in every batch.
    bool f32_pieces = x_dtype == ROCML_F32 && w_dtype == ROCML_F32 && out_dtype == ROCML_F32 && k % 4 == 0 && ldx % 4 == 0 &&
                      ldw % 4 == 0 && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0);
    if (f32_pieces && algo == ALGO_AUTO) {
        SplitPlan plan{defer, deferred_splits, RowScale{}, max_splits >= 1 && max_splits < 16 ? max_splits : 16};
        const float *xf = (const float*)x, *wf = (const float*)w;
        float* of = (float*)out;
        int rc;
#define F32_BY_EPI(fn, ...)                                                                  \
        (epi == EPI_ACC ? fn<EPI_ACC>(__VA_ARGS__) : epi == EPI_SWIGLU ? fn<EPI_SWIGLU>(__VA_ARGS__) \
         : epi == EPI_RELUGLU ? fn<EPI_RELUGLU>(__VA_ARGS__) : fn<EPI_F32>(__VA_ARGS__))
        if (m <= 32) rc = F32_BY_EPI(launch_f32_rows, xf, ldx, wf, ldw, of, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
        else rc = F32_BY_EPI(launch_f32_tile, xf, ldx, wf, ldw, of, ldo, m, n, k, workspace, workspace_bytes, plan, stream);
#undef F32_BY_EPI
        if (rc) return rc;
        ROCML_CHECK_LAUNCH("gemm");
        return 0;
    }
    ROCML_REQUIRE(!relu2, "gemm: the squared-rectifier epilogue goes with the matrix-core kernels (K and row strides multiples of 8)");
    // plain kernel; the gated epilogue runs as a second kernel over a 32-bit product in the workspace
    void* dst = out;
    int dst_ld = ldo, dst_dtype = out_dtype;
    if (gated) {
        ROCML_REQUIRE(workspace && workspace_bytes >= (long long)m * n * (long long)sizeof(float),
                      "gemm: the gated epilogue needs %lld bytes of workspace", (long long)m * n * 4);
        dst = workspace;
        dst_ld = n;
        dst_dtype = ROCML_F32;
    }
    if (x_dtype == ROCML_F32 && w_dtype == ROCML_F32 && dst_dtype == ROCML_F32) {
        launch_gemm_tile<float, float, float>(x, ldx, w, ldw, dst, dst_ld, m, n, k, accumulate, stream);
    } else if (bf16_in && dst_dtype == ROCML_F32) {
        launch_gemm_tile<bf16_t, bf16_t, float>(x, ldx, w, ldw, dst, dst_ld, m, n, k, accumulate, stream);
    } else if (bf16_in && dst_dtype == ROCML_BF16) {
        launch_gemm_tile<bf16_t, bf16_t, bf16_t>(x, ldx, w, ldw, dst, dst_ld, m, n, k, 0, stream);
    } else {
        return rocml_fail("gemm: unsupported type triple x=%d w=%d out=%d", x_dtype, w_dtype, out_dtype);
    }
    if (gated) {
        long long total = (long long)m * (n / 2);
        if (out_dtype == ROCML_F32)
            swiglu_pairs_kernel<float><<<ceil_div(total, 256), 256, 0, stream>>>((const float*)dst, (float*)out, ldo, m, n / 2, epilogue == 2);
        else
            swiglu_pairs_kernel<bf16_t><<<ceil_div(total, 256), 256, 0, stream>>>((const float*)dst, (bf16_t*)out, ldo, m, n / 2, epilogue == 2);
    }
    ROCML_CHECK_LAUNCH("gemm");
    return 0;
}

#include "gemm_heads.h"

// A batch of small products that share their shapes: out_b[M, N] = x_b[M, K] * w_b[N, K]^T for
// b = 0 .. batch-1, operands and results `batch_*` elements apart (the heads of a layer: x and out
// are column ranges of wider matrices, w is [batch, N, K]).  32-bit accumulation by fused
// multiply-add in K order for every type; x may be 32-bit while w is bfloat16.
// gate (may be null): 32-bit [M, ldg] with the heads side by side, batch_g apart: out = product * sigmoid(gate).
// gate_one: one gate number per head instead of one per column.
ROCML_EXPORT int rocml_gemm_batched(const void* x, int x_dtype, int ldx, long long batch_x, const void* w, int w_dtype,
                                    int ldw, long long batch_w, void* out, int out_dtype, int ldo, long long batch_o,
                                    int batch, int m, int n, int k, const float* gate, int ldg, long long batch_g,
                                    int gate_one, hipStream_t stream) {
    ROCML_REQUIRE(batch > 0 && batch < 65536 && m >= 0 && n > 0 && k > 0, "gemm_batched: bad sizes batch=%d M=%d N=%d K=%d", batch, m, n, k);
    ROCML_REQUIRE(ldx >= k && ldw >= k && ldo >= n && batch_x >= 0 && batch_w >= 0 && batch_o >= 0,
                  "gemm_batched: row strides (%d, %d, %d) below (K, K, N) or a negative batch stride", ldx, ldw, ldo);
    ROCML_REQUIRE(ceil_div(m, GT_BM) < 65536, "gemm_batched: too many rows %d", m);
    ROCML_REQUIRE(!gate || ldg >= (gate_one ? 1 : n), "gemm_batched: gate rows of %d numbers for N=%d", ldg, n);
    if (m == 0) return 0;
    // The matrix cores: bfloat16 weights [batch, N, K] without gaps, operands that 16-byte loads reach.
    int x_align = x_dtype == ROCML_F32 ? 4 : 8;
    bool mfma = w_dtype == ROCML_BF16 && out_dtype == ROCML_BF16 && ldw == k && batch_w == (long long)n * k && k % 8 == 0 &&
                ldx % x_align == 0 && batch_x % x_align == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
    if (mfma) {
        bool few = m <= 16;
        dim3 grid(few ? ceil_div(n, 32) : ceil_div(n, GH_BN), few ? 1 : ceil_div(m, GH_BM), batch);
#define GH(TX, G)                                                                                        \
        if (few) gemm_heads_few_rows_kernel<TX, bf16_t, G><<<grid, 256, 0, stream>>>(                    \
            (const TX*)x, ldx, (int)batch_x, (const bf16_t*)w, (bf16_t*)out, ldo, (int)batch_o, m, n, k, gate, ldg, (int)batch_g, gate_one); \
        else gemm_heads_mfma_kernel<TX, bf16_t, G><<<grid, 256, 0, stream>>>(                            \
            (const TX*)x, ldx, (int)batch_x, (const bf16_t*)w, (bf16_t*)out, ldo, (int)batch_o, m, n, k, gate, ldg, (int)batch_g, gate_one)
        if (x_dtype == ROCML_F32) { if (gate) { GH(float, true); } else { GH(float, false); } }
        else { if (gate) { GH(bf16_t, true); } else { GH(bf16_t, false); } }
#undef GH
        ROCML_CHECK_LAUNCH("gemm_batched");
        return 0;
    }
    ROCML_REQUIRE(!gate, "gemm_batched: the gate goes with the matrix-core kernel (bfloat16 weights and output, K a multiple of 8)");
#define GB(TX, TW, TO) launch_gemm_tile_batched<TX, TW, TO>(x, ldx, batch_x, w, ldw, batch_w, out, ldo, batch_o, batch, m, n, k, stream)
    if (x_dtype == ROCML_F32 && w_dtype == ROCML_F32 && out_dtype == ROCML_F32) GB(float, float, float);
    else if (x_dtype == ROCML_F32 && w_dtype == ROCML_BF16 && out_dtype == ROCML_BF16) GB(float, bf16_t, bf16_t);
    else if (x_dtype == ROCML_BF16 && w_dtype == ROCML_BF16 && out_dtype == ROCML_BF16) GB(bf16_t, bf16_t, bf16_t);
    else if (x_dtype == ROCML_BF16 && w_dtype == ROCML_BF16 && out_dtype == ROCML_F32) GB(bf16_t, bf16_t, float);
    else return rocml_fail("gemm_batched: unsupported type triple x=%d w=%d out=%d", x_dtype, w_dtype, out_dtype);
#undef GB
    ROCML_CHECK_LAUNCH("gemm_batched");
    return 0;
}

// The queries of a latent attention for at most 16 rows (latent_queries_kernel): out_h[M, 0 .. N) = q_h[M, 0 .. K) * w_h[N, K]^T and
// out_h[M, N .. N + rot_part) = the rotated numbers q_h[M, offset ..) of which the first dims turn.  q is 32-bit, w and out bfloat16.
ROCML_EXPORT int rocml_latent_queries(const float* q, int ldq, int q_stride, const void* w, void* out, int ldo, int o_stride, int heads,
                                      int m, int n, int k, int offset, int rot_part, int dims, const float* cos_t, const float* sin_t,
                                      int pairing, hipStream_t stream) {
    ROCML_REQUIRE(heads > 0 && heads < 65536 && m >= 0 && m <= 16 && n > 0 && k > 0 && rot_part >= 0 && dims >= 0 && dims % 2 == 0 && dims <= rot_part,
                  "latent_queries: bad sizes heads=%d M=%d N=%d K=%d part=%d dims=%d", heads, m, n, k, rot_part, dims);
    ROCML_REQUIRE(offset >= 0 && k <= q_stride && offset + rot_part <= q_stride && n + rot_part <= o_stride && ldq >= heads * q_stride && ldo >= heads * o_stride,
                  "latent_queries: a head does not hold its parts");
    ROCML_REQUIRE(k % 8 == 0 && ldq % 4 == 0 && q_stride % 4 == 0 && (uintptr_t)q % 16 == 0 && (uintptr_t)w % 16 == 0,
                  "latent_queries: rows and weights in 16-byte pieces are needed (K=%d ldq=%d)", k, ldq);
    ROCML_REQUIRE(pairing == 0 || pairing == 1, "latent_queries: pairing %d (0: halves, 1: neighbours)", pairing);
    ROCML_REQUIRE(q && w && out && (dims == 0 || (cos_t && sin_t)), "latent_queries: a pointer is missing");
    if (m == 0) return 0;
    latent_queries_kernel<<<dim3(ceil_div(n, 32) + 1, 1, heads), 256, 0, stream>>>(q, ldq, q_stride, (const bf16_t*)w, (bf16_t*)out, ldo, o_stride, m, n, k,
                                                                                   offset, rot_part, dims, cos_t, sin_t, pairing);
    ROCML_CHECK_LAUNCH("latent_queries");
    return 0;
}
