// x[M, N] += a[M, K] . w[N, K]^T (+ bias) for up to 16 rows, on packed weights, in one pass:
// the product that closes a mixer or a feed-forward adds itself to the residual stream and
// leaves, beside the stream, what the norm that follows needs of it.
//
// A block owns 16 (or 32, or 8) rows of w (as many columns of x) and the whole of k: its waves take equal runs of
// k, each with one MFMA accumulator; LDS adds the waves' sums in ascending order of k, the
// block adds them to its columns of x (float32, in place) and writes for every row of x the
// sum of the squares of its new values: sums[block][16], and x * norm_w in bfloat16, the rows
// of the rmsnorm that follows without their scale.  The product that takes norm(x) as its
// activations (gemm_skinny_lds_bf16.hip, PRODUCE_UNSCALED) multiplies these rows, adds the blocks'
// sums in ascending order and applies 1 / rms to its result: no other pass over x and no kernel
// between the two products.  Nothing here depends on what else runs: the order of every addition is
// fixed by N, K and the number of waves.
//
// HALF a strip a block: for matrices of few rows (N / 16 blocks fill half the compute units or less) a block takes 8 rows of w.
// What bounds such a product is what a unit can have on its way: [2048, 8192] at one row streams 33.5 MB in 10.5 us on 128 units
// and in 9.0 on 256 (8 rows: 11.2 -> 9.8).  The packed layout has 8 rows of a step as runs of 128 bytes, whole cache lines.
//
// (With k divided over blocks instead, as the few-row product with partial sums does, a row of x
// is complete only after a kernel boundary, and the norm has to be a kernel of its own: at 8
// rows two such kernels were 9.6 of a layer's 102 us.)
//
// Weights: llogos_pack_weights' layout, [N / 64][K / 32][4 strips][64 lanes] fragments of 16
// bytes; strip s of a 64-row group is every fourth KB of the group's run.  Activations: each
// wave copies the rows of a for its own run of k (rows beyond M: zero) through its own part of
// LDS; with at most 16 rows that is at most as many bytes as the weights, and they come from
// the L2.  A block with 16 waves holds 86 to 102 KB of LDS (the waves' copies and their sums).
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kResidualRows = 16;      // rows of a (tokens) at most

// AHEAD: MFMA steps (32 values of k) whose operands a wave asks for together.  HALF: the block owns half a strip.
template <int WAVES, int RB, bool HALF, int AHEAD>
__global__ __launch_bounds__(WAVES * kWave) void gemm_residual_kernel(
        float* __restrict__ x, int ldx, float* __restrict__ sums, bf16_t* __restrict__ unscaled, int ldu,
        const float* __restrict__ norm_w, const bf16_t* __restrict__ a, int lda,
        const u32x4* __restrict__ wp, const float* __restrict__ bias, int M, int N, int K) {
    static_assert(!HALF || RB == 1, "half a strip or whole ones");
    constexpr int kLoads = HALF ? AHEAD / 2 : AHEAD;     // loads of weights of a strip for AHEAD steps
    constexpr int kActRow = AHEAD * 32 + 8;              // bf16 of a wave's LDS row: AHEAD steps and 16 bytes of padding (rows 4 banks apart)
    constexpr int kRowLanes = AHEAD * 4, kLoadRows = kWave / kRowLanes;   // lanes that copy a row of activations, rows a load
    __shared__ float red[WAVES][RB][4][kWave];
    __shared__ __attribute__((aligned(16))) bf16_t acts[WAVES][kResidualRows][kActRow];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int r = lane & 15, g = lane >> 4;
    const int half = HALF ? blockIdx.x & 1 : 0;
    const int strip0 = HALF ? blockIdx.x >> 1 : blockIdx.x * RB;   // the block's RB strips of 16 rows of w follow one another
    const int steps = (K + 31) / 32;
    const int s_begin = (int)((long long)steps * wave / WAVES), s_end = (int)((long long)steps * (wave + 1) / WAVES);
    const u32x4* wsrc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int strip = strip0 + rb;
        wsrc[rb] = wp + ((size_t)(strip >> 2) * steps * 4 + (strip & 3)) * kWave + (HALF ? g * 16 + half * 8 + (r & 7) : lane);
    }
    const bool strip_ok[2] = {true, RB == 2 && (strip0 + 1) * 16 < N};
    // Activations: a wave copies the AHEAD steps' values of k of a few rows with one load (AHEAD * 4 lanes a row,
    // whole cache lines), through registers into its own rows of LDS, and reads its MFMA operands from
    // there.  (Loading the operands themselves, 16 rows x 64 bytes a step, asked for twice the lines: the
    // 8B down projection took 23.0 us at 8 rows, 20.6 without its activations, 20.9 with this copy.)
    const int copies = (M + kLoadRows - 1) / kLoadRows;
    const int cr = lane / kRowLanes, cl = lane % kRowLanes;
    const bf16_t* asrc = a + (size_t)cr * lda + cl * 8;
    const int k_end = min(K, s_end * 32);

    // HALF: a load brings the block's 8 rows of two steps, those of the second one in the operand's rows 8 to 15.  The operand is
    // multiplied with the activations of either step, into sums of their own: rows 0 to 7 of the first and 8 to 15 of the second count.
    f32x4 acc[RB], second = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 wf[2][kLoads][RB];
    uint4 af[2][kResidualRows / kLoadRows];
    auto fetch = [&](int buf, int s0) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j)
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const int s = HALF ? s0 + 2 * j + (r >> 3) : s0 + j;
                u32x4 v = {0, 0, 0, 0};
                if (s < s_end && strip_ok[rb]) v = __builtin_nontemporal_load(wsrc[rb] + (size_t)s * (4 * kWave));
                wf[buf][j][rb] = v;
            }
#pragma unroll
        for (int q = 0; q < kResidualRows / kLoadRows; ++q) {
            uint4 t = make_uint4(0, 0, 0, 0);
            if (q < copies && kLoadRows * q + cr < M && s0 * 32 + cl * 8 < k_end)
                t = *reinterpret_cast<const uint4*>(asrc + (size_t)(kLoadRows * q) * lda + s0 * 32);
            af[buf][q] = t;
        }
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int q = 0; q < kResidualRows / kLoadRows; ++q)
            *reinterpret_cast<uint4*>(&acts[wave][kLoadRows * q + cr][cl * 8]) = af[buf][q];
        // the rows are this wave's own: its lanes exchange them through LDS in program order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            const uint4 t = *reinterpret_cast<const uint4*>(&acts[wave][r][j * 32 + g * 8]);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                f32x4& to = HALF && (j & 1) ? second : acc[rb];
                to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[buf][HALF ? j / 2 : j][rb]),
                                                             __builtin_bit_cast(bf16x8, t), to, 0, 0, 0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // What the sums are added to: asked for behind the first weights, there long before it is needed.
    constexpr int kCols = HALF ? 8 : 16;                 // columns of x a strip of this block
    const int m = threadIdx.x / kCols, c = threadIdx.x % kCols;
    float x_old[RB], b_old[RB], nw[RB];
    if (s_begin < s_end) fetch(0, s_begin);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int n = HALF ? blockIdx.x * 8 + c : (strip0 + rb) * 16 + c;
        const bool in = m < M && n < N;
        x_old[rb] = in ? x[(size_t)m * ldx + n] : 0.f;
        b_old[rb] = in && bias ? bias[n] : 0.f;
        nw[rb] = in && unscaled ? norm_w[n] : 0.f;
    }
    for (int s = s_begin; s < s_end; s += 2 * AHEAD) {
        if (s + AHEAD < s_end) fetch(1, s + AHEAD);
        multiply(0);
        if (s + 2 * AHEAD < s_end) fetch(0, s + 2 * AHEAD);
        if (s + AHEAD < s_end) multiply(1);
    }

    // acc[rb][i]: column 16 (strip0 + rb) + 4 g + i of x, row r; HALF: column 8 blockIdx.x + 4 (g & 1) + i
    if (HALF && g >= 2) acc[0] = second;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][rb][i][lane] = acc[rb][i];
    __syncthreads();
    if (threadIdx.x >= kResidualRows * kCols) return;
    const int src_lane = (c >> 2) * 16 + m, i = c & 3;
    float sq = 0.f;                                      // of this thread's row over the block's columns
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        if (!strip_ok[rb]) continue;
        float v = 0.f, w2 = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            v += red[w][rb][i][src_lane];
            if (HALF) w2 += red[w][rb][i][src_lane + 32];
        }
        if (HALF) v += w2;
        const int n = HALF ? blockIdx.x * 8 + c : (strip0 + rb) * 16 + c;
        if (m < M && n < N) {
            const float y = x_old[rb] + (v + b_old[rb]);
            x[(size_t)m * ldx + n] = y;
            sq += y * y;
            if (unscaled) unscaled[(size_t)m * ldu + n] = f32_to_bf16(y * nw[rb]);
        }
    }
    // the lanes of a row are neighbours: a fixed tree of additions
#pragma unroll
    for (int o = kCols / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o, kWave);
    if (c == 0) sums[(size_t)blockIdx.x * kResidualRows + m] = sq;
}

// strips_per_block: 1 or 2 strips of 16 rows of w a block (two, of 4 or 8 waves, share a wave's copy of the activations and halve
// the number of blocks), or 0: half a strip.  sums: float32 [blocks][16], blocks = ceil(ceil(N / 16) / strips_per_block)
// or 2 ceil(N / 16), written whole (rows from M on hold 0): a block's sum of squares of each row of x over its 8, 16 or 32
// columns.  unscaled (optional, with norm_w [N]): bfloat16 [M][ldu] = x * norm_w of the new x, the rows of an rmsnorm that
// still lack their scale.
LLOGOS_EXPORT int llogos_gemm_residual_bf16(float* x, int ldx, float* sums, void* unscaled, int ldu, const float* norm_w,
                                            const void* act, int lda, const void* packed_w, const float* bias,
                                            int M, int N, int K, int waves, int strips_per_block, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || ldx < N || lda < K || x == nullptr || sums == nullptr) return LLOGOS_BAD_ARGUMENT;
    if (unscaled != nullptr && (norm_w == nullptr || ldu < N)) return LLOGOS_BAD_ARGUMENT;
    if (M > kResidualRows || (K % 8) || (lda % 8) || ((uintptr_t)act % 16) || ((uintptr_t)packed_w % 16))
        return LLOGOS_UNSUPPORTED;
    const int strips = (N + 15) / 16;
    const u32x4* W = (const u32x4*)packed_w;
    const bf16_t* A = (const bf16_t*)act;
#define GO(WAVES, RB, HALF, AHEAD) gemm_residual_kernel<WAVES, RB, HALF, AHEAD><<<HALF ? 2 * strips : (strips + RB - 1) / RB, WAVES * kWave, 0, stream>>>( \
        x, ldx, sums, (bf16_t*)unscaled, ldu, norm_w, A, lda, W, bias, M, N, K)
    if (strips_per_block == 1 && waves == 4) GO(4, 1, false, 4);
    else if (strips_per_block == 1 && waves == 8) GO(8, 1, false, 4);
    else if (strips_per_block == 1 && waves == 16) GO(16, 1, false, 4);
    else if (strips_per_block == 2 && waves == 4) GO(4, 2, false, 4);
    else if (strips_per_block == 2 && waves == 8) GO(8, 2, false, 4);
    else if (strips_per_block == 0 && waves == 8) GO(8, 1, true, 8);
    else if (strips_per_block == 0 && waves == 16) GO(16, 1, true, 4);
    else return LLOGOS_BAD_ARGUMENT;
#undef GO
    return LLOGOS_LAUNCH_CHECK();
}
