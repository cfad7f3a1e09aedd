// out[M, N] = a[M, K] . w[N, K]^T for more than 64 rows (prompts, steps of many sequences) on the matrix cores, with the weights in their packed
// order (llogos_pack_weights in gemm_skinny_lds_bf16.hip: blocks of 64 rows, steps of 32 k, fragments of 16 rows x 32 k).
// The kernel is tile_body in gemm_tiles.h; here are its entry points and what cuts a product into tiles.
//
//  * v_mfma_f32_16x16x32_bf16, rows of w first: a lane's four sums are consecutive rows of w for one token.  At the power limit, which is
//    what bounds a long product on this GPU, it does more than v_mfma_f32_32x32x16_bf16 (half the accumulator traffic a product):
//    8,192^3 in tiles of 256 x 256, zeros / random operands, us: 605 / 796 with 32x32x16, 572 / 715 with this one.
//  * A block is 4 waves, one a SIMD, each 64 rows of w (one packed block) by all of the tile's 64 to 256 tokens: w goes straight from memory
//    into the registers of the one wave that needs it, and only the activations go through LDS.  A stage of 64 k of a 256 x 256 tile so writes
//    32 KB to LDS and reads 128, where tiles with both operands in LDS on eight waves wrote 64 and read 192, more than LDS serves in the time
//    of the stage's products.
//  * A ring of four stages, in LDS and in registers: while one is multiplied the three after it are on their way.  The activations are copied
//    straight into LDS by buffer loads (rows of 128 bytes, the eight 16-byte pieces swizzled).  Two things had kept such rings one stage
//    deep: __syncthreads waits for every copy in flight (so a raw barrier here, and a wait for the copies that are due), and after a global_load_lds the
//    compiler waits for all loads at the next use of anything (the buffer form does not count as a flat access).
//  * One barrier a stage, a few products behind the last reads of a buffer, so that these have come back and the wait for them is short.
//    Products, reads and loads are written in issue order and pinned.  Loads past the last stage lie out of the buffer's range and
//    bring zeros: the loop has no tail.
//  * Results go through LDS so that whole lines are stored, non-temporally: kept in the L2 they push out the operands that the XCD's other
//    blocks share (8,192^3 765 -> 721 us).
//  * Blocks are numbered so that the 32 that run on an XCD are about 8 x 4 neighbouring tiles (tiles_place).
//  * Tiles of 64 to 256 tokens, blocks along k (float32 partial sums [parts][M][N] that the consumer adds), and the last round of blocks in tiles
//    of half the height, by a cost fitted to measurements (tiles_choose).
//  * Measured (us, weights from memory, in turn with other products; the tiles on eight waves of 32x32x16 products with both operands copied
//    through registers -> these, the library between): 2,048 tokens, 28,672 x 4,096 with SwiGLU 407 (380) 362, 4,096 x 14,336 in two parts
//    215 (217) 184, 4,096 x 4,096 70 (62) 63, 6,144 x 4,096 96 (81) 89; 5,003 tokens, 34,816 x 5,120 with SwiGLU 1,492 (1,541) 1,355,
//    5,120 x 17,408 800 (1,044) 680; 300 tokens, 28,672 x 4,096 with SwiGLU (86) 73; 65 tokens, 4,096 x 14,336 in eight parts (49) 28.  8,192^3:
//    1.54 PFLOP/s random, 1.92 zeros.
//  * Epilogues: plain (+ bias) in bfloat16 or float32; added to a float32 result in place; SwiGLU for a matrix packed with gate_rows; the activations of
//    two-matrix feed-forwards in bfloat16 (a float32 result and a kernel of its own took 50 us more a layer at 2,500 rows of 21,504 values:
//    215 MB written and read; a pass of that prompt and 16 steps 25,113 -> 24,461 us).
#include "gemm_tiles.h"

// What tiles of 64, 96, .. 256 tokens take, in microseconds: a launch, a round of blocks, a stage of 64 k, what a stage takes longer when
// every unit works, a MB of results (gated: a MB per 1,024 x 1,024 rows and tokens), a MB of weights; rounds and weights side by side but for a
// share of the shorter.  Fitted to 25,000 launches of 65 to 16,384 rows of 33 matrices ([512, 4,096] to [32,768, 2,048]) in 1 to 8 parts, and to
// 2,800 gated ones of 15 ([2,816, 896] to [57,344, 8,192]); rms 4 to 6 % from 128 tokens a tile on, 7 to 10 % below.  The height it chooses takes
// 0.2 to 0.7 % longer than the best of them on average, gated 0.5 % (a fit to three gated matrices took 3 %, and for up to 256 rows of
// [4,096, 768] and [9,728, 1,024] 1.2 to 2 times as long).
struct TilesTimes { double start, round, stage, busy, result, weight, both; };
static const TilesTimes kTilesPlain[7] = {
    {3.56, 0.73, 0.431, 0.062, 0.034, 0.118, 0.91}, {3.57, 1.98, 0.462, 0.127, 0.017, 0.109, 0.88}, {0.11, 6.19, 0.554, 0.182, 0.049, 0.144, 0.48},
    {0.59, 7.03, 0.667, 0.168, 0.059, 0.168, 0.31}, {0.15, 9.28, 0.732, 0.289, 0.034, 0.156, 0.21}, {0.22, 10.28, 0.852, 0.337, 0.035, 0.126, 0.22},
    {0.0, 11.24, 0.972, 0.395, 0.049, 0.119, 0.20}};
static const TilesTimes kTilesGated[7] = {
    {3.43, 0.0, 0.437, 0.099, 0.0, 0.106, 1.0}, {3.65, 0.0, 0.578, 0.031, 0.168, 0.075, 1.0}, {0.48, 4.24, 0.683, 0.087, 0.181, 0.050, 1.0},
    {0.44, 6.96, 0.710, 0.144, 0.104, 0.045, 1.0}, {0.94, 9.22, 0.712, 0.322, 0.0, 0.028, 1.0}, {1.40, 10.05, 0.818, 0.396, 0.0, 0.018, 1.0},
    {1.56, 11.23, 0.934, 0.455, 0.0, 0.014, 1.0}};

static double tiles_cost(int rows, int M, int N, int K, int parts, int units, bool gated) {
    const TilesTimes& t = (gated ? kTilesGated : kTilesPlain)[rows / 2 - 2];
    const double tiles = (double)((M + 16 * rows - 1) / (16 * rows)) * ((N + 255) / 256) * parts;
    const double rounds = ceil(ceil(tiles / 8.0) / (units / 8.0)), busy = tiles / (rounds * units);
    const int per = (K / kStageK + parts - 1) / parts, whole = (per + kRing - 1) / kRing * kRing;
    const double work = rounds * (t.round + whole * (t.stage + t.busy * busy)), weights = (double)N * K * 2e-6 * t.weight;
    return t.start + fmax(work, weights) + t.both * fmin(work, weights) + (double)M * N * (gated ? 1e-6 : 4e-6 * parts) * t.result;
}

struct TilesChoice { int rows, rows_last, n_full; double cost; };

// The cheapest cut of a product in `parts` parts of k: all tiles of one height, or of 256 tokens with the last round of blocks in tiles of 128
// (2,048 x 28,672 x 4,096 gated, three rounds and a half: 356 us all of 256, 353 cut; 2,048 x 34,816 x 5,120, four rounds and a quarter: 566 in the best
// one height, 538 cut).
static TilesChoice tiles_choose(int M, int N, int K, int parts, int units, bool gated) {
    const int n_tiles = (N + 255) / 256;
    TilesChoice best{16, 0, n_tiles, 1e30};
    for (int rows = 4; rows <= 16; rows += 2) {
        const double cost = tiles_cost(rows, M, N, K, parts, units, gated);
        if (cost < best.cost) best = TilesChoice{rows, 0, n_tiles, cost};
    }
    const int m16 = (M + 255) / 256;
    const int whole = (int)((long long)n_tiles * m16 * parts / units * units / ((long long)m16 * parts));          // row tiles in whole rounds
    if (whole > 0 && whole < n_tiles) {
        const double cost = tiles_cost(16, M, whole * 256, K, parts, units, gated) + tiles_cost(8, M, N - whole * 256, K, parts, units, gated);
        if (cost < best.cost) best = TilesChoice{16, 8, whole, cost};
    }
    return best;
}

static int tiles_launch(TilesCall c, int out_dtype, int epilogue, int token_tiles, int units) {
    c.rows_last = c.n_full = 0;
    if (token_tiles == 0) {
        const TilesChoice t = tiles_choose(c.M, c.N, c.K, c.parts, units, epilogue == EPI_SWIGLU);
        c.rows = t.rows, c.rows_last = t.rows_last, c.n_full = t.n_full;
    } else {
        c.rows = token_tiles <= 4 ? 4 * token_tiles : token_tiles;
    }
    if (epilogue == EPI_SWIGLU) return out_dtype == DT_BF16 ? tiles_gated_bf16(c) : tiles_gated_f32(c);
    if (epilogue == EPI_ADD) return tiles_add_f32(c);
    if (epilogue == EPI_RELU2) return tiles_relu2_bf16(c);
    if (epilogue == EPI_XIELU) return tiles_xielu_bf16(c);
    return out_dtype == DT_BF16 ? tiles_plain_bf16(c) : tiles_plain_f32(c);
}

// a: bfloat16 [M][lda]; packed_w: llogos_pack_weights of w [N][K]; out [parts][M][ldo] bfloat16 or float32.
// epilogue 0: out = a . w^T (+ bias [N]); 1: w's 16-row strips alternate gate and up rows, out is
// [M][N / 2] = silu(gate) * up, or with limit >= 0 the form of tiles_gated (no bias, one part); 2: out (float32) += a . w^T (no bias,
// one part).  parts > 1: float32 partial sums over ranges of k, part_stride
// elements apart, no bias.  token_tiles: 0: chosen here for a GPU of compute_units; 1 .. 4: tiles of 64 times as many tokens; 6, 10, 14: of 16
// times as many.  K must be a multiple of 64 and of more than one part every one must hold at least two stages of 64.
LLOGOS_EXPORT int llogos_gemm_tiles_bf16(void* out, int out_dtype, const void* a, int lda, const void* packed_w,
                                         const float* bias, int M, int N, int K, int ldo, long long part_stride,
                                         int epilogue, int parts, int token_tiles, int compute_units, float limit, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || out == nullptr || a == nullptr || packed_w == nullptr) return LLOGOS_BAD_ARGUMENT;
    if (out_dtype != DT_BF16 && out_dtype != DT_F32) return LLOGOS_BAD_ARGUMENT;
    if (epilogue < EPI_PLAIN || epilogue > EPI_ADD) return LLOGOS_BAD_ARGUMENT;
    if (epilogue == EPI_ADD && (out_dtype != DT_F32 || bias != nullptr || parts != 1)) return LLOGOS_BAD_ARGUMENT;
    // (a wave's loads count bytes from its tile's first row, or its block of w, in 31 bits)
    if ((K % kStageK) || (lda % 8) || lda < K || lda > 1 << 21 || ((uintptr_t)a % 16) || ((uintptr_t)packed_w % 16)) return LLOGOS_UNSUPPORTED;
    if (epilogue == EPI_SWIGLU && ((N % 32) || bias != nullptr || ldo < N / 2 || parts != 1)) return LLOGOS_BAD_ARGUMENT;
    if (epilogue != EPI_SWIGLU && ldo < N) return LLOGOS_BAD_ARGUMENT;
    if (token_tiles < 0 || (token_tiles > 4 && token_tiles != 6 && token_tiles != 10 && token_tiles != 14)) return LLOGOS_BAD_ARGUMENT;
    if (parts < 1 || compute_units < 1) return LLOGOS_BAD_ARGUMENT;
    if (parts > 1 && (out_dtype != DT_F32 || bias != nullptr || part_stride < (long long)M * ldo)) return LLOGOS_BAD_ARGUMENT;
    if (parts > 1 && (K / kStageK) / parts < 2) return LLOGOS_UNSUPPORTED;          // every part holds two stages or more
    TilesCall c{};
    c.out = out, c.a = a, c.wp = packed_w, c.bias = bias, c.lda = lda, c.M = M, c.N = N, c.K = K, c.ldo = ldo, c.parts = parts;
    c.part_stride = part_stride, c.limit = limit, c.stream = stream;
    return tiles_launch(c, out_dtype, epilogue, token_tiles, compute_units);
}

// out [M][ldo] bfloat16 = act(a . w^T) in one part, kinds of activation.h: the square of relu, or xIELU with its two numbers.
LLOGOS_EXPORT int llogos_gemm_tiles_activated_bf16(void* out, const void* a, int lda, const void* packed_w, int M, int N, int K, int ldo, int kind, float act_a,
                                                   float act_b, int compute_units, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || out == nullptr || a == nullptr || packed_w == nullptr || lda < K || ldo < N || compute_units < 1) return LLOGOS_BAD_ARGUMENT;
    if (kind != ACT_RELU2 && kind != ACT_XIELU) return LLOGOS_UNSUPPORTED;
    if ((K % kStageK) || (lda % 8) || lda > 1 << 21 || ((uintptr_t)a % 16) || ((uintptr_t)packed_w % 16)) return LLOGOS_UNSUPPORTED;
    TilesCall c{};
    c.out = out, c.a = a, c.wp = packed_w, c.lda = lda, c.M = M, c.N = N, c.K = K, c.ldo = ldo, c.parts = 1;
    c.limit = act_a, c.act_b = act_b, c.stream = stream;
    return tiles_launch(c, DT_BF16, kind == ACT_RELU2 ? EPI_RELU2 : EPI_XIELU, 0, compute_units);
}

// Microseconds that a product in `parts` parts is expected to take in the tiles that token_tiles = 0 chooses.
LLOGOS_EXPORT double llogos_gemm_tiles_cost(int M, int N, int K, int parts, int compute_units) {
    if (M <= 0 || N <= 0 || K < kStageK || parts < 1 || compute_units < 1) return 1e30;
    return tiles_choose(M, N, K, parts, compute_units, false).cost;
}

// Tokens a tile that token_tiles = 0 chooses, less the half tiles of a last round.
LLOGOS_EXPORT int llogos_gemm_tiles_height(int M, int N, int K, int parts, int compute_units, int gated) {
    if (M <= 0 || N <= 0 || K < kStageK || parts < 1 || compute_units < 1) return LLOGOS_BAD_ARGUMENT;
    return 16 * tiles_choose(M, N, K, parts, compute_units, gated != 0).rows;
}
