// out[M, N] = a[M, K] . w[N, K]^T for prompts of some hundred rows, with the weights in their packed order
// (llogos_pack_weights in gemm_skinny_lds_bf16.hip): tiles of 64, 128 or 192 tokens by 256 rows of w, whose stages of k are dealt
// out to several blocks where the tiles alone leave compute units idle.
//
//  * What bounds it: with so few rows a matrix is a tile or two of tokens high, and its row tiles (16 of 4,096 rows) fill a
//    fraction of the units; every unit then waits for its own chain of stages.  So the tile is as low as the rows need (64
//    tokens), and blocks along k fill the units: 70 rows of [4,096, 14,336] are 2 x 16 tiles in 8 parts.  The float32 partial
//    sums are the consumer's to add.
//  * v_mfma_f32_32x32x16_bf16, rows of w first: 4 waves, one a SIMD, 2 along the rows of w (128 each) by 2 along the tokens (TM x 32
//    each).  A wave's 4 + TM operands serve 4 TM products; the waves of gemm_tiles_bf16.hip, eight of 64 rows, read 2 + TM for
//    2 TM, which shows where TM is small (its tiles of 128 tokens were 5 % slower, those of 256 level).
//  * Stages of 64 values of k, two LDS buffers; copies go through registers, asked for two stages ahead and stored one
//    stage ahead, in LDS order as in gemm_tiles_bf16.hip (operands of w as 1 KB in lane order; activations as rows of 128 bytes
//    whose 16-byte pieces are swizzled).  One barrier a stage, between the third and the fourth sub-step of 16 k: the stores are
//    in the first three, the first reads of the next stage in the fourth.
//  * Sums are those of gemm_tiles_bf16.hip in the same parts, bit for bit.
//  * Measured (us, the library's product -> this one, whose parts are still to be added): 128 rows: [2,048, 2,048] 20.0 -> 11.2,
//    [3,072, 2,048] 20.1 -> 12.3, [4,096, 4,096] 21.5 -> 16.4, [7,168, 5,120] 33.4 -> 25.0, [5,120, 17,408] 150 -> 47; 256 rows:
//    [6,144, 4,096] 35.8 -> 25.1, [5,120, 5,120] 44.6 -> 24.5.  [4,096, 14,336]: 128 rows 44 (the few-row product) -> 33, 334 rows 61
//    (tiles of 128 tokens of gemm_tiles_bf16.hip in 4 parts) -> 53.
#include "gemm_tiles.h"

constexpr int kWavesN = 2, kWavesM = 2, kTileWaves = 4;
constexpr int kTileBlocks = 4;                         // packed blocks of 64 rows of w a tile: 256 rows
constexpr int kStageK = 64;
constexpr int kStageW = kTileBlocks * 64 * kStageK * 2;   // 32 KB

template <int N> __device__ __forceinline__ void short_wait_loads() {
    static_assert(N == 9 || N == 11 || N == 13, "a stage's copies but one");
    if (N == 9) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
    if (N == 11) asm volatile("s_waitcnt vmcnt(11)" ::: "memory");
    if (N == 13) asm volatile("s_waitcnt vmcnt(13)" ::: "memory");
}

template <int TM, typename TO>
__global__ __launch_bounds__(kTileWaves * kWave, 1) void gemm_tiles_short_kernel(
        TO* __restrict__ out, const bf16_t* __restrict__ a, int lda, const unsigned char* __restrict__ wp, int M, int N, int K, int ldo,
        size_t part_stride, int n_row_blocks, int m_tiles, int n_tiles, int parts) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    int m_tile, u;
    if (!tiles_place(m_tiles * n_tiles * parts, m_tiles, n_tiles * parts, blockIdx.x & 7, blockIdx.x >> 3, m_tile, u)) return;
    const int part = u / n_tiles, n_tile = u % n_tiles;
    // (the parts divide the stages evenly, as in gemm_tiles_bf16.hip)
    const int all = K / kStageK, stage_begin = (int)((long long)all * part / parts), stage_end = (int)((long long)all * (part + 1) / parts);
    out += (size_t)part * part_stride;
    constexpr int BM = kWavesM * TM * 32;
    constexpr int kStageBytes = kStageW + BM * kStageK * 2;
    constexpr int kPieces = 8 + 2 * TM;                                      // copies per wave and stage: 8 of w, 2 TM of the activations
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wn = wave & (kWavesN - 1), wm = wave / kWavesN;
    const int steps = K / 32, stages = stage_end - stage_begin;
    const int m0 = m_tile * BM;
    const int r32 = lane & 31, h = lane >> 5;

    const int w_block = min(n_tile * kTileBlocks + wave, n_row_blocks - 1);
    const unsigned char* w_src = wp + ((size_t)w_block * steps + 2 * stage_begin) * 4096 + (size_t)(r32 >> 4) * 1024 +
                                 (size_t)((r32 & 15) + 16 * h) * 16;
    const int w_dst = wave * 2 * 4096 + lane * 16;
    const bf16_t* a_src[2 * TM];
    const int a_dst = kStageW + wave * 2 * TM * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) {
        const int row = 8 * (wave * 2 * TM + i) + (lane >> 3), oct = (lane & 7) ^ ((row >> 1) & 7);
        a_src[i] = a + (size_t)min(m0 + row, M - 1) * lda + (size_t)stage_begin * kStageK + 8 * oct;
    }
    u32x4_t g[kPieces];
    auto fetch_one = [&](int c, int stage) {
        if (c < 8) g[c] = *reinterpret_cast<const u32x4_t*>(w_src + (size_t)stage * 2 * 4096 + (c >> 2) * 4096 + ((c >> 1) & 1) * 2048 + (c & 1) * 512);
        else g[c] = *reinterpret_cast<const u32x4_t*>(a_src[c - 8] + (size_t)stage * kStageK);
    };
    auto store_one = [&](int buf, int c) {
        unsigned char* base = lds + buf * kStageBytes;
        if (c < 8) *reinterpret_cast<u32x4_t*>(base + w_dst + c * 1024) = g[c];
        else *reinterpret_cast<u32x4_t*>(base + a_dst + (c - 8) * 1024) = g[c];
    };

    f32x16_t acc[TM][4];
#pragma unroll
    for (int tt = 0; tt < TM; ++tt)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[tt][rt][v] = 0.f;

    const int w_read = wn * 4 * 4096 + lane * 16;
    int a_read[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) a_read[j] = kStageW + (wm * TM * 32 + r32) * 128 + (((2 * j + h) ^ ((r32 >> 1) & 7)) * 16);
    struct Frags { bf16x8_t w[4]; bf16x8_t a[TM]; };
    // fragment i of sub-step j: 0 .. 3 rows of w, 4 .. 3 + TM tokens
    auto read_one = [&](Frags& f, int buf, int j, int i) {
        const unsigned char* base = lds + buf * kStageBytes;
        if (i < 4) f.w[i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(
            base + w_read + (i >> 1) * 8192 + (j >> 1) * 4096 + (2 * (i & 1) + (j & 1)) * 1024));
        else f.a[i - 4] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(base + a_read[j] + (i - 4) * 4096));
    };
    auto mfma = [&](const Frags& f, int i) {
        const int tt = i >> 2, rt = i & 3;
        acc[tt][rt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[rt], f.a[tt], acc[tt][rt], 0, 0, 0);
    };
    // A sub-step's 4 TM products with other work between them: the 4 + TM fragments of the sub-step that follows (of the next
    // buffer behind the last) and, in the first three, a third of the copies each: a piece is stored for the next stage (all but
    // the pieces asked for after it have arrived) and asked for again for the stage after next.
    constexpr int kReads = 4 + TM, kProducts = 4 * TM;
    auto sub = [&](const Frags& cur, Frags& nxt, int buf, int j, int far) {
        const int c0 = j < 3 ? kPieces * j / 3 : kPieces, c1 = j < 3 ? kPieces * (j + 1) / 3 : kPieces;
        const int ops = kReads + 2 * (c1 - c0);
#pragma unroll
        for (int i = 0; i < kProducts; ++i) {
            mfma(cur, i); SB();
#pragma unroll
            for (int o = 0; o < kReads + 12; ++o) {
                if (o < ops * i / kProducts || o >= ops * (i + 1) / kProducts) continue;
                if (o < kReads) read_one(nxt, j < 3 ? buf : buf ^ 1, (j + 1) & 3, o);
                else if (((o - kReads) & 1) == 0) { short_wait_loads<kPieces - 1>(); store_one(buf ^ 1, c0 + (o - kReads) / 2); }
                else fetch_one(c0 + (o - kReads) / 2, far);
                SB();
            }
        }
    };

    Frags f0, f1;
    // prologue: the first stage into buffer 0; the pieces of the second asked for in the order in which they are stored
#pragma unroll
    for (int c = 0; c < kPieces; ++c) fetch_one(c, 0);
#pragma unroll
    for (int c = 0; c < kPieces; ++c) store_one(0, c);
#pragma unroll
    for (int c = 0; c < kPieces; ++c) fetch_one(c, min(1, stages - 1));
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kReads; ++i) read_one(f0, 0, 0, i);
    SB();
    for (int s = 0; s + 1 < stages; ++s) {
        const int buf = s & 1, far = min(s + 2, stages - 1);                 // (past the end: the last stage again, never stored)
        sub(f0, f1, buf, 0, far);
        sub(f1, f0, buf, 1, far);
        sub(f0, f1, buf, 2, far);
        // the next stage is stored, and this one's last fragments are read: from here on the buffers have changed places
        __syncthreads();
        SB();
        sub(f1, f0, buf, 3, far);
    }
    {
        const int buf = (stages - 1) & 1;
        auto last = [&](const Frags& cur, Frags& nxt, int j) {
#pragma unroll
            for (int i = 0; i < kReads; ++i) read_one(nxt, buf, j + 1, i);
            SB();
#pragma unroll
            for (int i = 0; i < kProducts; ++i) { mfma(cur, i); SB(); }
        };
        last(f0, f1, 0); last(f1, f0, 1); last(f0, f1, 2);
#pragma unroll
        for (int i = 0; i < kProducts; ++i) { mfma(f1, i); SB(); }
    }

    const int strip0 = 8 * n_tile + 4 * wn;                                  // the wave's first 32 rows of w, counted in such (none is stored past N)
    const bool wide = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & (4 * sizeof(TO) - 1)) == 0;
#pragma unroll
    for (int tt = 0; tt < TM; ++tt) {
        const int token = m0 + 32 * (wm * TM + tt) + r32;
        if (token >= M) continue;
        TO* orow = out + (size_t)token * ldo;
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = 32 * (strip0 + rt) + 8 * q + 4 * h;
                const float* y = reinterpret_cast<const float*>(&acc[tt][rt]) + 4 * q;
                if (wide && n + 3 < N) {
                    if (sizeof(TO) == 2) {
                        uint2 pk;
                        pk.x = tiles_pack_bf16(y[0], y[1]);
                        pk.y = tiles_pack_bf16(y[2], y[3]);
                        *reinterpret_cast<uint2*>(orow + n) = pk;
                    } else {
                        *reinterpret_cast<float4*>(orow + n) = make_float4(y[0], y[1], y[2], y[3]);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < N) store_f32(orow + n + e, y[e]);
                }
            }
    }
}

template <int TM, typename TO>
static int launch_short(void* out, const void* a, int lda, const void* wp, int M, int N, int K, int ldo, long long part_stride, int parts,
                        hipStream_t stream) {
    const int n_row_blocks = (N + 63) / 64, n_tiles = (n_row_blocks + kTileBlocks - 1) / kTileBlocks, m_tiles = (M + 64 * TM - 1) / (64 * TM);
    const long long tiles = (long long)m_tiles * n_tiles * parts;
    if (tiles > 1 << 24) return LLOGOS_UNSUPPORTED;
    constexpr size_t smem = (size_t)2 * (kStageW + TM * 64 * kStageK * 2);
    static std::atomic<uint64_t> asked{0};
    const int code = allow_dynamic_lds((const void*)gemm_tiles_short_kernel<TM, TO>, (int)smem, asked);
    if (code != 0) return code;
    gemm_tiles_short_kernel<TM, TO><<<(unsigned)((tiles + 7) / 8 * 8), kTileWaves * kWave, smem, stream>>>(
        (TO*)out, (const bf16_t*)a, lda, (const unsigned char*)wp, M, N, K, ldo, (size_t)part_stride, n_row_blocks, m_tiles, n_tiles, parts);
    return LLOGOS_LAUNCH_CHECK();
}

// a: bfloat16 [M][lda]; packed_w: llogos_pack_weights of w [N][K], rows in their order; out [parts][M][ldo] float32 (or, in one
// part, bfloat16), part_stride elements apart.  token_tiles: 64 tokens times 1, 2 or 3.  K must be a multiple of 64, and every
// part must hold at least two stages of 64.
LLOGOS_EXPORT int llogos_gemm_tiles_short_bf16(void* out, int out_dtype, const void* a, int lda, const void* packed_w, int M, int N, int K,
                                               int ldo, long long part_stride, int parts, int token_tiles, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || out == nullptr || a == nullptr || packed_w == nullptr) return LLOGOS_BAD_ARGUMENT;
    if (out_dtype != DT_BF16 && out_dtype != DT_F32) return LLOGOS_BAD_ARGUMENT;
    if ((K % kStageK) || (lda % 8) || lda < K || ((uintptr_t)a % 16) || ((uintptr_t)packed_w % 16)) return LLOGOS_UNSUPPORTED;
    if (ldo < N || parts < 1 || token_tiles < 1 || token_tiles > 3) return LLOGOS_BAD_ARGUMENT;
    if (parts > 1 && (out_dtype != DT_F32 || part_stride < (long long)M * ldo)) return LLOGOS_BAD_ARGUMENT;
    if (parts > 1 && (K / kStageK) / parts < 2) return LLOGOS_UNSUPPORTED;
#define GO(TM) do { if (out_dtype == DT_BF16) return launch_short<TM, bf16_t>(out, a, lda, packed_w, M, N, K, ldo, part_stride, parts, stream); \
                    return launch_short<TM, float>(out, a, lda, packed_w, M, N, K, ldo, part_stride, parts, stream); } while (0)
    if (token_tiles == 1) GO(1);
    if (token_tiles == 2) GO(2);
    GO(3);
#undef GO
}
