// out[M, N] = a[M, K] . w[N, K]^T (+ bias[N]), all float32, every product and sum in 32 bits: the
// matrix product of the float32 engine, on v_mfma_f32_16x16x4f32.  That instruction is a chain of
// four fused multiply-adds in ascending slot order, one rounding each (checked bit by bit against
// fmaf, denormals too), so nothing is rounded more than by plain FMAs at twice their rate.
//
// Every output element is summed in one order, whatever the kernel and the step's row count:
//   part: 16 consecutive k, chained from 0 in the order k = e + 4 g, e = 0..3 outside, g = 0..3
//         inside (slot g of MFMA e holds element e of the four values at 4 g, so that a lane's
//         operands for four MFMAs are one 16-byte load);
//   mid:  the parts of 256 consecutive k, added in ascending order;
//   total: the mids in ascending order.
// So a row's result is the same bits alone and in any batch, and the rounding error of a sum over
// thousands of k grows with its blocks (16 + 16 + K / 256 additions deep) and not with K.
//
// One to four rows (gemm_f32_lanes_kernel) and few rows (gemm_f32_rows_kernel): bound by reading w once.
// In the second a block owns 16 or 32 rows of w and all of k; its waves take 256 k in turn straight from
// memory, a mid each, and LDS adds the mids in order.  Many rows: bound by the matrix cores (157 TFLOP/s at 2.4 GHz, of which no form
// reached more than 117); gemm_f32_ring_kernel where K is a multiple of 32, else gemm_f32_tiles_kernel: tiles of 128 x 64, 64 x 64 or 64 x 32
// through two LDS buffers of 32 k.
// Measured (us; before: plain FMAs in tiles of 64 x 64, up to 32 rows a wave for a few columns).  705 rows of the 1B
// sizes, these / tiles / ring: gate/up [16384, 2048] 1,507 / 478 / 436 (109 TFLOP/s), o [2048, 2048] about 390 / 70 / 62, down [2048, 8192] about
// 1,510 / 270 / 238, q/k/v [3072, 2048] 448 / 108 / 97.  2 rows: gate/up 28.3 -> 28.6 (4.7 TB/s), head [128256, 2048] 209 -> 180
// (5.8 TB/s).  Distance from 64 bits at k = 8192: 1.5e-7 of the result.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

// values k .. k + 3 of a row, zeros from K on; VEC: rows start at multiples of 16 bytes and K % 4 == 0
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* __restrict__ row, int k, int K) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        if (k < K) v = *reinterpret_cast<const f32x4*>(row + k);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) if (k + e < K) v[e] = row[k + e];
    }
    return v;
}

// four neighbouring columns of one row of the result
__device__ __forceinline__ void store4(float* __restrict__ out, const float* __restrict__ bias, f32x4 v, int m, int n, int N, int ldo, bool vec) {
    if (vec && n + 3 < N) {
        if (bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += bias[n + r];
        }
        *reinterpret_cast<f32x4*>(out + (size_t)m * ldo + n) = v;
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (n + r < N) out[(size_t)m * ldo + n + r] = bias ? v[r] + bias[n + r] : v[r];
}

// part = the chain over one block of 16 k: lane (i = lane & 15, g = lane >> 4) holds k = 4 g .. 4 g + 3 of row i of either operand
__device__ __forceinline__ f32x4 chain16(f32x4 w, f32x4 a) {
    f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) p = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], a[e], p, 0, 0, 0);
    return p;
}

// WAVES waves a block; MT tiles of 16 rows of a and NS strips of 16 rows of w.  PL blocks of 16 k are asked for at once (8 KB of w a
// wave at MT = NS = 1): in flight enough to stream w from memory with 16 waves a compute unit.
template <int WAVES, int MT, int NS, bool VEC>
__global__ __launch_bounds__(WAVES * 64) void gemm_f32_rows_kernel(
        float* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w,
        const float* __restrict__ bias, int M, int N, int K, int lda, int ldo, int vec_out) {
    constexpr int TILES = MT * NS, PL = TILES == 1 ? 8 : 4, OWN = (TILES + WAVES - 1) / WAVES;
    __shared__ f32x4 mids[WAVES][TILES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16 * NS, m0 = blockIdx.y * 16 * MT;
    const float* wrow[NS];
    const float* arow[MT];
#pragma unroll
    for (int s = 0; s < NS; ++s) wrow[s] = w + (size_t)min(n0 + 16 * s + i, N - 1) * K;
#pragma unroll
    for (int t = 0; t < MT; ++t) arow[t] = a + (size_t)min(m0 + 16 * t + i, M - 1) * lda;
    f32x4 total[OWN];
#pragma unroll
    for (int o = 0; o < OWN; ++o) total[o] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int groups = (K + 255) / 256;
    for (int g0 = 0; g0 < groups; g0 += WAVES) {                 // the same trips for every wave: the barriers match
        const int grp = g0 + wave;
        f32x4 mid[NS][MT];
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int t = 0; t < MT; ++t) mid[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (grp < groups) {
#pragma unroll 1
            for (int p0 = 0; p0 < 16; p0 += PL) {
                const int k0 = grp * 256 + p0 * 16;
                if (k0 >= K) break;
                f32x4 wv[PL][NS], av[PL][MT];
#pragma unroll
                for (int p = 0; p < PL; ++p) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) wv[p][s] = load4<VEC>(wrow[s], k0 + 16 * p + 4 * g, K);
#pragma unroll
                    for (int t = 0; t < MT; ++t) av[p][t] = load4<VEC>(arow[t], k0 + 16 * p + 4 * g, K);
                }
#pragma unroll
                for (int p = 0; p < PL; ++p)
                    if (k0 + 16 * p < K) {
#pragma unroll
                        for (int s = 0; s < NS; ++s)
#pragma unroll
                            for (int t = 0; t < MT; ++t) mid[s][t] += chain16(wv[p][s], av[p][t]);
                    }
            }
        }
        if (g0 > 0) __syncthreads();                             // the mids of the trip before have been read
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int t = 0; t < MT; ++t) mids[wave][s * MT + t][lane] = mid[s][t];
        __syncthreads();
        const int here = min(WAVES, groups - g0);
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const int tile = wave + o * WAVES;
            if (tile < TILES)
                for (int j = 0; j < here; ++j) total[o] += mids[j][tile][lane];
        }
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int tile = wave + o * WAVES;
        if (tile >= TILES) continue;
        const int m = m0 + 16 * (tile % MT) + i, n = n0 + 16 * (tile / MT) + 4 * g;
        if (m < M) store4(out, bias, total[o], m, n, N, ldo, vec_out != 0);
    }
}

// The fewest rows by plain multiply-adds: a wave takes COLS rows of w, a lane 16 consecutive k of them and of every row of a at a
// time; it chains a part in the order above, sixteen neighbouring lanes hold the parts of a mid, and the mids are added in
// order.  No wave waits for another, and a matrix of few rows has a wave for each where the kernel above has one block for 16:
// 1 row, us, that kernel -> this one: [2048, 8192] 27.3 -> 15.6 (4.3 TB/s), [4096, 14336] 49.7 -> 40.4 (5.8), [2048, 2048] 8.5 -> 5.8,
// [16, 16384] 42.9 -> 14.4, [50000, 768] 40.0 -> 26.8, [1000, 1001] 14.4 -> 5.4.
template <int MR, int COLS, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_lanes_kernel(
        float* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w,
        const float* __restrict__ bias, int M, int N, int K, int lda, int ldo) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n0 = (blockIdx.x * 4 + wave) * COLS, m0 = blockIdx.y * MR;
    if (n0 >= N) return;
    float total[MR];                                            // lane c: the totals of column n0 + c
#pragma unroll
    for (int m = 0; m < MR; ++m) total[m] = 0.f;
    for (int k0 = 0; k0 < K; k0 += 1024) {
        f32x4 av[MR][4];
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int g = 0; g < 4; ++g) av[m][g] = load4<VEC>(a + (size_t)min(m0 + m, M - 1) * lda, k0 + 16 * lane + 4 * g, K);
#pragma unroll 1
        for (int c = 0; c < COLS; ++c) {
            f32x4 wv[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) wv[g] = load4<VEC>(w + (size_t)min(n0 + c, N - 1) * K, k0 + 16 * lane + 4 * g, K);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                float part = 0.f, mid = 0.f, sum = total[m];
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int g = 0; g < 4; ++g) part = fmaf(wv[g][e], av[m][g][e], part);
#pragma unroll
                for (int j = 0; j < 16; ++j) mid += __shfl(part, (lane & 48) + j, kWave);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float m4 = __shfl(mid, 16 * g, kWave);
                    if (k0 + 256 * g < K) sum += m4;
                }
                total[m] = lane == c ? sum : total[m];
            }
        }
    }
    if (lane < COLS && n0 + lane < N) {
#pragma unroll
        for (int m = 0; m < MR; ++m)
            if (m0 + m < M) out[(size_t)(m0 + m) * ldo + n0 + lane] = bias ? total[m] + bias[n0 + lane] : total[m];
    }
}

// Tiles of TM rows of a x TN rows of w, four waves in two rows and two columns.  Rows of 32 k lie in LDS at a stride of 40 words:
// 16 rows x 4 columns of 16 bytes are then read without bank conflicts.
template <int TM, int TN, bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_f32_tiles_kernel(
        float* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w,
        const float* __restrict__ bias, int M, int N, int K, int lda, int ldo, int vec_out, int m_tiles, int n_tiles) {
    constexpr int KS = 32, LD = 40, MT = TM / 32, NT = TN / 32, COPIES = (TM + TN) * (KS / 4) / 256;
    __shared__ __align__(16) float lds[2][(TM + TN) * LD];
    // an XCD (every eighth block) takes neighbouring tiles, the rows of a fastest: its L2 keeps the rows of w
    const int blocks = m_tiles * n_tiles, per = blocks / 8, more = blocks % 8, xcd = blockIdx.x & 7;
    const int tile = xcd * per + min(xcd, more) + (blockIdx.x >> 3);
    const int m0 = (tile % m_tiles) * TM, n0 = (tile / m_tiles) * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, g = lane >> 4;
    const int wm = (wave & 1) * (TM / 2), wn = (wave >> 1) * (TN / 2);

    const float* src[COPIES];
    int dst[COPIES];
#pragma unroll
    for (int c = 0; c < COPIES; ++c) {
        const int piece = tid + 256 * c, row = piece >> 3, col = (piece & 7) * 4;
        src[c] = row < TM ? a + (size_t)min(m0 + row, M - 1) * lda : w + (size_t)min(n0 + row - TM, N - 1) * K;
        dst[c] = row * LD + col;
    }
    const int col = (tid & 7) * 4;
    // a stage is asked for two stages ahead (one: gate/up 477 us against 459, q/k/v 123 against 115); past K the last values are
    // read again (a load under a condition would make every wait one for all loads) and zeros are stored
    f32x4 ahead[2][COPIES];
    auto load = [&](f32x4 (&to)[COPIES], int k) {
#pragma unroll
        for (int c = 0; c < COPIES; ++c)
            to[c] = VEC ? *reinterpret_cast<const f32x4*>(src[c] + min(k + col, K - 4)) : load4<false>(src[c], k + col, K);
    };
    auto store = [&](const f32x4 (&from)[COPIES], float* to, int k) {
        const bool in = !VEC || k + col < K;
#pragma unroll
        for (int c = 0; c < COPIES; ++c) *reinterpret_cast<f32x4*>(to + dst[c]) = in ? from[c] : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    load(ahead[0], 0);
    load(ahead[1], KS);
    store(ahead[0], lds[0], 0);
    __syncthreads();

    f32x4 mid[NT][MT], total[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) mid[n][m] = total[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto stage = [&](int k0, int at) {                           // `at`: the stage's buffer, 0 or 1
        load(ahead[at], k0 + 2 * KS);
        const float* buf = lds[at];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (k0 + 16 * p >= K) break;
            f32x4 av[MT], wv[NT];
#pragma unroll
            for (int m = 0; m < MT; ++m) av[m] = *reinterpret_cast<const f32x4*>(buf + (wm + 16 * m + i) * LD + 16 * p + 4 * g);
#pragma unroll
            for (int n = 0; n < NT; ++n) wv[n] = *reinterpret_cast<const f32x4*>(buf + (TM + wn + 16 * n + i) * LD + 16 * p + 4 * g);
            f32x4 part[NT][MT];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        part[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[n][e], av[m][e], e ? part[n][m] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            const bool fold = ((k0 / 16 + p) & 15) == 15;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int m = 0; m < MT; ++m) mid[n][m] += part[n][m];
            if (fold) {
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int m = 0; m < MT; ++m) { total[n][m] += mid[n][m]; mid[n][m] = f32x4{0.f, 0.f, 0.f, 0.f}; }
            }
        }
        store(ahead[at ^ 1], lds[at ^ 1], k0 + KS);              // the other buffer was last read before the barrier behind it
        __syncthreads();
    };
    for (int k0 = 0; k0 < K; k0 += 2 * KS) {
        stage(k0, 0);
        if (k0 + KS < K) stage(k0 + KS, 1);
    }
    const bool open = (((K + 15) / 16) & 15) != 0;              // parts since the last fold
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            f32x4 v = total[n][m];
            if (open) v += mid[n][m];
            const int row = m0 + wm + 16 * m + i;
            if (row < M) store4(out, bias, v, row, n0 + wn + 16 * n + 4 * g, N, ldo, vec_out != 0);
        }
}

// Many rows, K a multiple of 32: the same sums with the matrix cores kept at work by each wave alone.  4 waves, WM along the rows of a by WN along the
// rows of w, each 16 MT x 16 NT of the result.  A ring of four stages of 32 k in LDS, filled by buffer loads (rows of 128 bytes, their eight 16-byte
// pieces swizzled); one raw barrier a stage, in front of it a wait for the copies of the next stage alone.  A step of 16 k is MT NT chains of four
// products; between them, pinned, one to a product: the additions of the step before to its mids (a chain's last product is long done by then), the
// reads of the next step's operands, the copies of the stage after next but one.  Eight stages are written out, so that the additions to the total
// stand in one place; stages past K bring zeros, and zeros change no sum.
template <int MT, int NT, int WM, int WN>
__global__ __launch_bounds__(256, 2) void gemm_f32_ring_kernel(
        float* __restrict__ out, const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias, int M, int N, int K,
        int lda, int ldo, int vec_out, int m_tiles, int n_tiles) {
#ifdef __HIP_DEVICE_COMPILE__
    constexpr int BM = 16 * MT * WM, BN = 16 * NT * WN, ROWS = BM + BN, BUF = ROWS * 128, RING = 4;
    constexpr int COPIES = (ROWS / 8 + 3) / 4, LEAST = ROWS / 8 / 4;         // of 8 rows a wave and stage; what every wave has of them
    constexpr int TILES = MT * NT, READS = MT + NT, PRODUCTS = 4 * TILES;
    static_assert(WM * WN == 4 && ROWS % 8 == 0, "four waves");
    // (the additions behind the products are assembly, for which the compiler adds no waits: a chain's last product has another tile's product and
    // the next step's first one behind it when it is read, 64 clocks; with one tile a wave nothing would stand between them)
    static_assert(TILES >= 2, "additions one step behind their products");
    extern __shared__ __attribute__((aligned(1024))) unsigned char f32_lds[];
    const int tiles = m_tiles * n_tiles, per = tiles >> 3, more = tiles & 7, xcd = blockIdx.x & 7;
    const int tile = xcd * per + min(xcd, more) + (blockIdx.x >> 3);
    const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15, g = lane >> 4;
    const int wm = (wave % WM) * 16 * MT, wn = (wave / WM) * 16 * NT;
    const int stages = K / 32;

    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(a + (size_t)m0 * lda), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, 0x7fffffff, 0x00020000);
    unsigned off[COPIES];
#pragma unroll
    for (int c = 0; c < COPIES; ++c) {
        const int row = 8 * (4 * c + wave) + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
        off[c] = (row < BM ? (unsigned)min(row, M - 1 - m0) * (unsigned)(4 * lda) : (unsigned)min(row - BM, N - 1 - n0) * (unsigned)(4 * K)) + 16 * piece;
    }
    auto copy = [&](int slot, int c, int stage, unsigned past) {
        const int q = 4 * c + wave;                                          // (the same for a whole wave)
        if (ROWS / 8 % 4 != 0 && c == COPIES - 1 && q >= ROWS / 8) return;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(q < BM / 8 ? a_rsrc : w_rsrc, (__attribute__((address_space(3))) void*)(f32_lds + slot * BUF + q * 1024), 16,
                                                 off[c] | past, stage * 128, 0, 0);
    };
    auto past_end = [&](int stage) { return stage < stages ? 0u : 0x80000000u; };
    int at[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) at[p] = i * 128 + (((4 * p + g) ^ ((i >> 1) & 7)) * 16);
    struct Frags { f32x4 a[MT], w[NT]; };
    auto read_one = [&](Frags& f, int slot, int p, int r) {
        const unsigned char* base = f32_lds + slot * BUF + at[p];
        if (r < MT) f.a[r] = *reinterpret_cast<const f32x4*>(base + (wm + 16 * r) * 128);
        else f.w[r - MT] = *reinterpret_cast<const f32x4*>(base + (BM + wn + 16 * (r - MT)) * 128);
    };
    float mid[NT][MT][4], total[NT][MT][4];
    f32x4 part[2][NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            part[0][n][m] = part[1][n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < 4; ++v) mid[n][m][v] = total[n][m][v] = 0.f;
        }
    auto meet = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // step p of the stage in `slot`, of the products cur; next: the step behind it
    auto step = [&](const Frags& cur, Frags& next, int slot, int p, int stage) {
        const unsigned past = past_end(stage + 3);
        f32x4 (&now)[NT][MT] = part[p];
        const f32x4 (&before)[NT][MT] = part[p ^ 1];
#pragma unroll
        for (int x = 0; x < PRODUCTS; ++x) {
            const int e = x / TILES, n = x % TILES / MT, m = x % MT;
            now[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.w[n][e], cur.a[m][e], e ? now[n][m] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            {                                                                // one addition a product: tile x / 4, value x % 4
                const int tn = x / 4 / MT, tm = x / 4 % MT;
                asm volatile("v_add_f32 %0, %1, %0" : "+v"(mid[tn][tm][x % 4]) : "v"(before[tn][tm][x % 4]));
            }
            if (p == 0) {
#pragma unroll
                for (int c = COPIES * x / PRODUCTS; c < COPIES * (x + 1) / PRODUCTS; ++c) copy((slot + 3) & 3, c, stage + 3, past);
#pragma unroll
                for (int r = READS * x / PRODUCTS; r < READS * (x + 1) / PRODUCTS; ++r) read_one(next, slot, 1, r);
            } else if (x == TILES - 1) {
                // every operand of this buffer is here (the products above took them), and so are this wave's copies of the next stage
                asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * LEAST) : "memory");
                meet();
            } else if (x >= TILES) {
#pragma unroll
                for (int r = READS * (x - TILES) / (PRODUCTS - TILES); r < READS * (x - TILES + 1) / (PRODUCTS - TILES); ++r) read_one(next, (slot + 1) & 3, 0, r);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int c = 0; c < COPIES; ++c) copy(s, c, s, past_end(s));
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * LEAST) : "memory");
    meet();
    Frags f0, f1;
#pragma unroll
    for (int r = 0; r < READS; ++r) read_one(f0, 0, 0, r);
    int s = 0;
    do {                                                         // 256 k
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            step(f0, f1, j & 3, 0, s + j);
            if (j == 0) {                                        // the last step of the 256 k before is in: their mids are whole
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int v = 0; v < 4; ++v) { total[n][m][v] += mid[n][m][v]; mid[n][m][v] = 0.f; }
            }
            step(f1, f0, j & 3, 1, s + j);
        }
        s += 8;
    } while (s < stages);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // copies still on their way into LDS
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = total[n][m][e] + (mid[n][m][e] + part[1][n][m][e]);
            const int row = m0 + wm + 16 * m + i;
            if (row < M) store4(out, bias, v, row, n0 + wn + 16 * n + 4 * g, N, ldo, vec_out != 0);
        }
#endif
}

namespace {

constexpr double kUnitFlops = 157.3e12 / 256;               // of one compute unit

// Seconds that the two kernels take, fitted to sweeps of 1 to 2,048 rows over eight matrices.  Tiles: a stage of 32 k takes a block that is
// alone on its compute unit 0.35 us beside its products; blocks that share a unit hide that, and share the matrix cores, which the
// kernel keeps busy 70 % of the time.
double tiles_cost(double M, double N, double K, int tm, int tn, double units) {
    const double blocks = ceil(M / tm) * ceil(N / tn), tile = tm * (double)tn * 2 / kUnitFlops * (tn == 32 ? 1.6 : 1.4);
    const double together = tn == 32 ? 4 : tm == 64 ? 3 : 2;
    const double busy = ceil(blocks / units) * tile * K, waits = ceil(blocks / (units * together)) * (tile * K + K / 32 * 0.35e-6);
    return (busy > waits ? busy : waits) + 3e-6;
}

// Microseconds of the ring: forms 9 to 12.  A stage of 32 k of a block alone on its compute unit takes `alone`, of each of `together` blocks that
// share one `shared` (the matrix cores at 72 to 75 % of their rate, whatever runs beside them).  Fitted to 64 to 1,024 rows of six matrices, within 6 %.
struct RingForm { int tm, tn, together; double alone, shared; };
constexpr RingForm kRing[4] = {{64, 64, 2, 0.66, 0.573}, {64, 32, 3, 0.46, 0.288}, {48, 64, 2, 0.556, 0.48}, {80, 64, 2, 0.89, 0.746}};

double ring_cost(double M, double N, double K, const RingForm& f, double units) {
    const int blocks = (int)ceil(ceil(M / f.tm) * ceil(N / f.tn) / units), rest = blocks % f.together;
    const double stage = (blocks - rest) * f.shared + (rest ? (rest * f.shared > f.alone ? rest * f.shared : f.alone) : 0.0);
    return (5.0 + ceil(K / 256) * 8 * stage) * 1e-6;
}

// 17 rows and more by the few-row kernel: what its blocks ask of the caches (their strips of w and the rows of a, once a block), at the rates
// that the three forms were measured at, with compute units idle while a last round of blocks runs.
double rows_cost(double M, double N, double K, int mt, int ns, double units) {
    const double blocks = ceil(N / (16 * ns)) * ceil(M / (16 * mt));
    const double spread = blocks < units ? blocks / units : blocks / units / ceil(blocks / units);
    return blocks * (ns + mt) * 64 * K / ((ns == 2 ? 5.3e12 : mt == 4 ? 6.7e12 : 9.5e12) * units / 256) / spread + 4e-6;      // (rates of 256 units)
}

// Rows of w a wave of the lanes' kernel takes, 0 where the few-row kernel is ahead: matrices whose blocks of 16 rows leave units idle
// or whose k gives those blocks' waves little to do (1 row, us, few-row kernel and this one: [6144, 4096] 30 and 22, [8192, 8192] 60 and
// 58, [16384, 2048] 27.3 and 26.7, [12288, 4096] 44 and 46, [128256, 2048] 177 and 196; 2 rows: [8192, 8192] 61 and 70, [24576, 1024] 24
// and 22).  Rows that are not aligned are read value by value, which the few-row kernel's lanes do at sixteen places of a line
// each; there it is ahead from 5 rows on ([50000, 769], 1 row 127 and 87, 4 rows 132 and 119; [3000, 4099] 39 and 41).
int lanes_cols(int M, int N, int K, bool vec) {
    if (!vec) return M > 4 ? 0 : (N <= 2048 ? 1 : (N > 16384 ? 8 : (K <= 1024 ? 2 : 0)));
    if (M > 2) return 0;
    if (N <= 3584 || (M == 1 && K <= 1024)) return 1;
    if (N <= (M == 1 ? 8192 : 6144)) return 2;
    return (M == 1 && N <= 16384 && K <= 2048) || (M == 2 && K <= 1024) ? 4 : 0;
}

}  // namespace

#define ROWS(W, MT, NS) do { \
        const dim3 grid((N + 16 * NS - 1) / (16 * NS), (M + 16 * MT - 1) / (16 * MT)); \
        if (vec) gemm_f32_rows_kernel<W, MT, NS, true><<<grid, W * 64, 0, stream>>>(out, a, w, bias, M, N, K, lda, ldo, vec_out); \
        else gemm_f32_rows_kernel<W, MT, NS, false><<<grid, W * 64, 0, stream>>>(out, a, w, bias, M, N, K, lda, ldo, vec_out); \
    } while (0)
#define LANES(MR, COLS, VEC) gemm_f32_lanes_kernel<MR, COLS, VEC><<<dim3((N + 4 * COLS - 1) / (4 * COLS), (M + MR - 1) / MR), 256, 0, stream>>>( \
        out, a, w, bias, M, N, K, lda, ldo)
#define TILES(TM, TN) do { \
        const int mt = (M + TM - 1) / TM, nt = (N + TN - 1) / TN; \
        if (vec) gemm_f32_tiles_kernel<TM, TN, true><<<mt * nt, 256, 0, stream>>>(out, a, w, bias, M, N, K, lda, ldo, vec_out, mt, nt); \
        else gemm_f32_tiles_kernel<TM, TN, false><<<mt * nt, 256, 0, stream>>>(out, a, w, bias, M, N, K, lda, ldo, vec_out, mt, nt); \
    } while (0)

#define RING(MT, NT, WM, WN) do { \
        const int mt = (M + 16 * MT * WM - 1) / (16 * MT * WM), nt = (N + 16 * NT * WN - 1) / (16 * NT * WN); \
        constexpr int smem = 4 * 128 * 16 * (MT * WM + NT * WN); \
        static std::atomic<uint64_t> asked{0}; \
        const int code = allow_dynamic_lds((const void*)gemm_f32_ring_kernel<MT, NT, WM, WN>, smem, asked); \
        if (code != 0) return code; \
        gemm_f32_ring_kernel<MT, NT, WM, WN><<<mt * nt, 256, smem, stream>>>(out, a, w, bias, M, N, K, lda, ldo, vec_out, mt, nt); \
    } while (0)

// form: 0 chosen by the costs above; 1 to 4 the few-row kernel with 16, 32, 64 rows of a or 64 rows of a and 32 of w a block; 5 to 7 tiles of
// 64 x 32, 64 x 64, 128 x 64; 8 the lanes' kernel; 9 to 12 the ring's tiles of 64 x 64, 64 x 32, 48 x 64, 80 x 64
LLOGOS_EXPORT int llogos_gemm_f32(float* out, const float* a, const float* w, const float* bias,
                                  int M, int N, int K, int lda, int ldo, int form, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || lda < K || ldo < N || form < 0 || form > 12) return LLOGOS_BAD_ARGUMENT;
    const bool vec = (K & 3) == 0 && (lda & 3) == 0 && (((uintptr_t)a | (uintptr_t)w) & 15) == 0;
    const int vec_out = (ldo & 3) == 0 && ((uintptr_t)out & 15) == 0;
    const int cols = lanes_cols(M, N, K, vec), units = device_units();
    if (form == 0 && cols) form = 8;
    // (the ring counts a tile's bytes from its first row in 31 bits, and asks for whole stages of aligned rows)
    const bool ring = vec && K % 32 == 0 && lda <= 1 << 22 && K <= 1 << 22;
    if (form > 8 && !ring) return LLOGOS_UNSUPPORTED;
    if (form == 0) {
        const double cost[5] = {0, 0, rows_cost(M, N, K, 2, 1, units), rows_cost(M, N, K, 4, 1, units), rows_cost(M, N, K, 4, 2, units)};
        form = M <= 16 ? 1 : 2;
        double least = cost[2];
        for (int f = 3; form > 1 && f <= (ring ? 12 : 7); ++f) {
            if (f == 5 && ring) f = 9;
            const double c = f < 5 ? cost[f] : f == 5 ? tiles_cost(M, N, K, 64, 32, units) : f == 6 ? tiles_cost(M, N, K, 64, 64, units)
                           : f == 7 ? tiles_cost(M, N, K, 128, 64, units) : ring_cost(M, N, K, kRing[f - 9], units);
            if (c < least) { least = c; form = f; }
        }
    }
    // 16 waves a block where a matrix has few blocks and enough of k for all of them
    const bool wide = K >= 16 * 256 && (N + 15) / 16 * ((M + 15) / 16) <= 2 * units;
    switch (form) {
        case 1: if (wide) ROWS(16, 1, 1); else ROWS(8, 1, 1); break;
        case 2: if (wide) ROWS(16, 2, 1); else ROWS(8, 2, 1); break;
        case 3: ROWS(8, 4, 1); break;
        case 4: ROWS(8, 4, 2); break;
        case 5: TILES(64, 32); break;
        case 6: TILES(64, 64); break;
        case 7: TILES(128, 64); break;
        case 9: RING(2, 2, 2, 2); break;
        case 10: RING(2, 1, 2, 2); break;
        case 11: RING(3, 1, 1, 4); break;
        case 12: RING(5, 1, 1, 4); break;
        default:
            if (vec && M == 1) { if (cols == 4) LANES(1, 4, true); else if (cols == 2) LANES(1, 2, true); else LANES(1, 1, true); }
            else if (vec) { if (cols == 4) LANES(2, 4, true); else if (cols == 2) LANES(2, 2, true); else LANES(2, 1, true); }
            else if (M == 1) { if (cols == 8) LANES(1, 8, false); else if (cols == 2) LANES(1, 2, false); else LANES(1, 1, false); }
            else if (M == 2) { if (cols == 8) LANES(2, 8, false); else if (cols == 2) LANES(2, 2, false); else LANES(2, 1, false); }
            else { if (cols == 8) LANES(4, 8, false); else if (cols == 2) LANES(4, 2, false); else LANES(4, 1, false); }
            break;
    }
    return LLOGOS_LAUNCH_CHECK();
}
