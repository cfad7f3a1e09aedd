// The products of experts chosen a token (moe.hip) with the matrices in their packed order: E matrices of N rows, a multiple of 64, packed as one
// of E N rows (llogos_pack_weights in gemm_skinny_lds_bf16.hip: blocks of 64 rows, steps of 32 k, strips of 16 rows x 32 k).  Sorted rows,
// segments and epilogues are those of moe.hip.
//   few rows  tiles of 16 sorted rows; a block of four waves owns a strip, its waves take 64 k in turn, and LDS adds their sums in order: the
//             sums of moe.hip's few-row form, bit for bit.  Bound by reading the matrices of the chosen experts.  A wave's load is one
//             whole KB of w, past the L2 (row-major it is sixteen half lines, which reach 5.4 to 5.9 TB/s whatever is in flight);
//             the four strips of a packed block fall to blocks of one XCD that start together, so that the 4 KB of a step are read from
//             memory at once.  16 experts of [7168, 4096], two a token, alone: 4 tokens 72 -> 62 us, 32 tokens (all) 162 -> 134 (7.0 TB/s;
//             strips in the grid's order 140; ordinary loads 152); [4096, 7168]: 71 -> 60 and 159 -> 135; 8 steps in flight a wave for 4: level or slower.
//   tiles     64 to 256 sorted rows x 256 rows of the matrix: tile_products of gemm_tiles.h on rows found through the order.  The number of
//             tiles is known on the device alone: the grid holds as many as there could be, and the blocks count them, choose their height and
//             share them out, so that an XCD's run of tiles is as long as the others'.
#include "gemm_tiles.h"
#include "moe.h"

template <typename TO>
__global__ __launch_bounds__(256) void moe_few_packed_kernel(TO* __restrict__ out, const bf16_t* __restrict__ a, const unsigned char* __restrict__ wp,
                                                             const int* __restrict__ order, const int* __restrict__ seg, int E, int top, int gather,
                                                             int N, int K, int lda, int act, float scale, const float* __restrict__ row_weight, float limit) {
    __shared__ float red[3][kWave][4];
    __shared__ int s_tile[3];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // block b of XCD x = b & 7 takes strip (j & 3) of the packed block x + 8 (j >> 2), j = b >> 3
    const int j = blockIdx.x >> 3, n0 = 64 * ((blockIdx.x & 7) + 8 * (j >> 2)) + 16 * (j & 3);
    if (n0 >= N) return;
    if (wave == 0) {
        int e, first, end;
        moe_find_tile(seg, E, 16, blockIdx.y, e, first, end);
        if (lane == 0) { s_tile[0] = e; s_tile[1] = first; s_tile[2] = end; }
    }
    __syncthreads();
    const int e = __builtin_amdgcn_readfirstlane(s_tile[0]), m0 = s_tile[1], m_end = s_tile[2];
    if (e < 0) return;
    const int c = lane & 15, g = lane >> 4;
    const int m = m0 + c;
    const int src = min(m, m_end - 1);                       // (rows past the segment's end are read as its last one: their sums go nowhere)
    const bf16_t* arow = a + (size_t)(gather ? order[src] / top : src) * lda + 8 * g;
    const int steps = K / 32;
    const unsigned char* w = wp + (((size_t)e * N + n0) >> 6) * steps * 4096 + ((n0 >> 4) & 3) * 1024 + lane * 16;
    auto row_frag = [&](int step) { return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(arow + 32 * step)); };
    auto w_frag = [&](int step) { return __builtin_bit_cast(bf16x8_t, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(w + (size_t)step * 4096))); };
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int AHEAD = 4;                                 // the rows are asked for in front of w, which comes back behind them
    int s = 2 * wave;
    auto step = [&](int i) { return s + 8 * (i >> 1) + (i & 1); };           // the wave's i-th step of 32 k from here
    for (; step(AHEAD - 1) < steps; s += 4 * AHEAD) {
        bf16x8_t wf[AHEAD], af[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) af[i] = row_frag(step(i));
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) wf[i] = w_frag(step(i));
        SB();
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], af[i], acc, 0, 0, 0);
    }
    for (; s < steps; s += 8)
        for (int half = 0; half < 2 && s + half < steps; ++half)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_frag(s + half), row_frag(s + half), acc, 0, 0, 0);
    if (wave > 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave - 1][lane][r] = acc[r];
    }
    __syncthreads();
    if (wave > 0 || m >= m_end) return;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        v[r] = ((acc[r] + red[0][lane][r]) + red[1][lane][r]) + red[2][lane][r];
        if (act == 1) { v[r] = fmaxf(v[r], 0.f); v[r] *= v[r]; }
        if (act < 2) v[r] *= scale;
    }
    const int n = n0 + 4 * g;
    if (act >= 2) {
        const float rw = row_weight ? row_weight[order[m]] : 1.0f;
        moe_store2(out + (size_t)m * (N / 2) + n / 2, moe_gated(v[0] * rw, v[1] * rw, act, limit) * scale, moe_gated(v[2] * rw, v[3] * rw, act, limit) * scale);
    } else moe_store4(out + (size_t)m * N + n, v[0], v[1], v[2], v[3]);
}

// How high the tiles are (64, 128, 192 or 256 sorted rows) is chosen here, where the segments are known: the height whose rounds of blocks take
// least, a round being round + stages (stage + busy x the share of the units that work) microseconds (gemm_tiles_bf16.hip: kTilesPlain).  From the
// average alone no height serves: 16 experts of [4096, 7168] with 125 rows on average, us in tiles of 128 / 192 / 256: even segments 248 / 169 /
// 224, uneven ones (Dirichlet 3) 244 / 328 / 215 (row-major 262 and 247).
struct MoeRound { float round, stage, busy; };
__device__ constexpr MoeRound kMoeRound[4] = {{4.2f, 0.543f, 0.f}, {5.1f, 0.577f, 0.154f}, {9.0f, 0.745f, 0.229f}, {10.6f, 0.996f, 0.292f}};

// For one whole wave: the height chosen of least .. most (units of 64 rows) and the tiles of all segments together in it.
__device__ __forceinline__ void moe_choose_height(const int* __restrict__ seg, int E, int least, int most, int n_tiles, int stages, int units, int& height, int& row_tiles) {
    const int lane = threadIdx.x & (kWave - 1);
    int tiles[4] = {0, 0, 0, 0};
    for (int e0 = 0; e0 < E; e0 += kWave) {
        const int rows = seg[min(e0 + lane + 1, E)] - seg[min(e0 + lane, E)];
#pragma unroll
        for (int h = 0; h < 4; ++h) tiles[h] += (rows + 64 * h + 63) / (64 * h + 64);
    }
    float cheapest = INFINITY;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) tiles[h] += __shfl_xor(tiles[h], o, kWave);
        if (h + 1 < least || h + 1 > most) continue;
        const float blocks = (float)tiles[h] * n_tiles, rounds = ceilf(ceilf(blocks * 0.125f) * 8.f / units);
        const float cost = rounds * (kMoeRound[h].round + stages * (kMoeRound[h].stage + kMoeRound[h].busy * blocks / (fmaxf(rounds, 1.f) * units)));
        if (cost < cheapest) { cheapest = cost; height = h + 1; row_tiles = tiles[h]; }
    }
}

template <int TM, int EPI, typename TO>
__device__ __forceinline__ void moe_tile(unsigned char* lds, TO* __restrict__ out, const bf16_t* __restrict__ a, const unsigned char* __restrict__ wp,
                                         const int* __restrict__ order, int top, int gather, int N, int K, int lda, int act, float scale,
                                         const float* __restrict__ row_weight, float limit, int e, int m0, int m_end, int n_tile) {
    const int n_blocks = N / 64, nb = n_tile * kTileBlocks + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    unsigned a_off[TM / 2];
#pragma unroll
    for (int i = 0; i < TM / 2; ++i) {
        const int row = tiles_a_row<TM>(i), src = min(m0 + row, m_end - 1);
        a_off[i] = (unsigned)(gather ? order[src] / top : src) * (unsigned)(lda * 2) + 16 * ((threadIdx.x & 7) ^ ((row >> 1) & 7));
    }
    f32x4_t acc[TM][4];
    tile_products<TM>(lds, acc, wp + ((size_t)e * n_blocks + min(nb, n_blocks - 1)) * (K / 32) * 4096, reinterpret_cast<const unsigned char*>(a), a_off, K / kStageK);
    TileEnd at{};
    at.m0 = m0, at.m_end = m_end, at.N = N, at.ldo = EPI == EPI_ROWS_GATED ? N / 2 : N, at.nb = nb, at.n_row_blocks = n_blocks;
    at.limit = act == 3 ? limit : -1.f, at.act = act, at.scale = scale, at.row_weight = row_weight, at.order = order;
    tile_store<TM, EPI, TO>(lds, acc, out, at);
}

template <int EPI, typename TO>
__global__ __launch_bounds__(kTileWaves * kWave, 1) void moe_tiles_packed_kernel(
        TO* __restrict__ out, const bf16_t* __restrict__ a, const unsigned char* __restrict__ wp, const int* __restrict__ order,
        const int* __restrict__ seg, int E, int top, int gather, int N, int K, int lda, int act, float scale, const float* __restrict__ row_weight, float limit,
        int least, int most, int units) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char moe_lds[];
    __shared__ int s_tile[5];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), n_tiles = (N + 255) / 256;
    if (wave == 0) {
        int height = least, row_tiles = 0, m_tile, n_tile = 0, e = -1, first = 0, end = 0;
        moe_choose_height(seg, E, least, most, n_tiles, K / kStageK, units, height, row_tiles);
        if (tiles_place(row_tiles * n_tiles, row_tiles, n_tiles, blockIdx.x & 7, blockIdx.x >> 3, m_tile, n_tile)) moe_find_tile(seg, E, 64 * height, m_tile, e, first, end);
        if (threadIdx.x == 0) { s_tile[0] = e; s_tile[1] = first; s_tile[2] = end; s_tile[3] = n_tile; s_tile[4] = height; }
    }
    __syncthreads();
    const int e = __builtin_amdgcn_readfirstlane(s_tile[0]), m0 = __builtin_amdgcn_readfirstlane(s_tile[1]), m_end = __builtin_amdgcn_readfirstlane(s_tile[2]);
    const int n_tile = __builtin_amdgcn_readfirstlane(s_tile[3]), height = __builtin_amdgcn_readfirstlane(s_tile[4]);
    if (e < 0) return;
#define MOE_TILE(TM) moe_tile<TM, EPI, TO>(moe_lds, out, a, wp, order, top, gather, N, K, lda, act, scale, row_weight, limit, e, m0, m_end, n_tile)
    if (height == 1) MOE_TILE(4);
    else if (height == 2) MOE_TILE(8);
    else if (height == 3) MOE_TILE(12);
    else MOE_TILE(16);
#undef MOE_TILE
}

struct MoePacked {
    void* out;
    const void* a;
    const void* wp;
    const int* order;
    const int* seg;
    int E, top, gather, P, N, K, lda, act;
    float scale;
    const float* row_weight;
    float limit;
    hipStream_t stream;
};

template <int EPI, typename TO>
static int launch_moe_tiles(const MoePacked& c, int least, int most, int units) {
    const long long row_tiles = (c.P + 64 * least - 1) / (64 * least) + c.E, blocks = (row_tiles * ((c.N + 255) / 256) + 7) / 8 * 8;
    if (blocks > 1 << 26) return LLOGOS_UNSUPPORTED;
    const int smem = tiles_lds_bytes(4 * most);
    static std::atomic<uint64_t> asked{0};
    const int code = allow_dynamic_lds((const void*)moe_tiles_packed_kernel<EPI, TO>, tiles_lds_bytes(16), asked);
    if (code != 0) return code;
    moe_tiles_packed_kernel<EPI, TO><<<(unsigned)blocks, kTileWaves * kWave, smem, c.stream>>>(
        (TO*)c.out, (const bf16_t*)c.a, (const unsigned char*)c.wp, c.order, c.seg, c.E, c.top, c.gather, c.N, c.K, c.lda, c.act, c.scale, c.row_weight, c.limit,
        least, most, units);
    return LLOGOS_LAUNCH_CHECK();
}

// llogos_moe_product_bf16 on the packed copy of w.  a has a_rows rows.  least 0: the few-row form; else tiles of 64 times least .. most (1 .. 4)
// sorted rows, whichever the segments make cheapest on a GPU of compute_units.  -2 for shapes these do not take: N no multiple of 64, K none of 32 (tiles: of 64).
LLOGOS_EXPORT int llogos_moe_product_packed_bf16(void* out, int out_dtype, const void* a, int a_rows, const void* wp, const int* order, const int* seg,
                                                 int E, int top, int gather, int P, int N, int K, int lda, int act, float scale,
                                                 const float* row_weight, float limit, int least, int most, int compute_units, hipStream_t stream) {
    if (P <= 0 || N <= 0 || K <= 0 || E <= 0 || top <= 0 || lda < K || a_rows <= 0 || act < 0 || act > 3 || (row_weight && act < 2) || (act == 3 && !(limit >= 0.f))) return LLOGOS_BAD_ARGUMENT;
    if ((out_dtype != DT_F32 && out_dtype != DT_BF16) || least < 0 || (least > 0 && (most < least || most > 4 || compute_units < 1))) return LLOGOS_BAD_ARGUMENT;
    if ((N % 64) || (K % (least ? kStageK : 32)) || (lda % 8) || ((uintptr_t)a % 16) || ((uintptr_t)wp % 16) || ((uintptr_t)out % 16)) return LLOGOS_UNSUPPORTED;
    // (a tile's loads count bytes from the first row of a in 31 bits)
    if (least && ((long long)a_rows * lda * 2 >= 1LL << 31)) return LLOGOS_UNSUPPORTED;
    const MoePacked c{out, a, wp, order, seg, E, top, gather, P, N, K, lda, act, scale, row_weight, limit, stream};
    if (least == 0) {
        const int row_tiles = (P + 15) / 16 + E;
        if (row_tiles > 65535) return LLOGOS_UNSUPPORTED;
        const dim3 grid((N / 64 + 7) / 8 * 32, row_tiles);
#define MOE_FEW(TO) moe_few_packed_kernel<TO><<<grid, 256, 0, stream>>>((TO*)out, (const bf16_t*)a, (const unsigned char*)wp, order, seg, E, top, gather, N, K, lda, act, scale, row_weight, limit)
        if (out_dtype == DT_F32) MOE_FEW(float); else MOE_FEW(bf16_t);
#undef MOE_FEW
        return LLOGOS_LAUNCH_CHECK();
    }
    if (act >= 2) return out_dtype == DT_BF16 ? launch_moe_tiles<EPI_ROWS_GATED, bf16_t>(c, least, most, compute_units) : launch_moe_tiles<EPI_ROWS_GATED, float>(c, least, most, compute_units);
    return out_dtype == DT_BF16 ? launch_moe_tiles<EPI_ROWS, bf16_t>(c, least, most, compute_units) : launch_moe_tiles<EPI_ROWS, float>(c, least, most, compute_units);
}
