// The tiled product for many rows on packed weights (gemm_tiles_bf16.hip): which block takes which tile, and one tile.
#pragma once
#include "activation.h"
#include "common.h"
#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

#define SB() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ uint32_t tiles_pack_bf16(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Which tile block j of XCD x takes, of `rows` token tiles x `cols` columns (a part of k and a row tile; the parts outermost):
// tiles are counted in bands of eight token tiles, a column of the band before the next, and every XCD takes a run of them, as
// long as the others' to one tile.  The 32 blocks that run on an XCD so are about 8 x 4 tiles of one part of k: they share
// their weights and their activations in its L2, and no XCD is left with a round of blocks more than the others.  (With
// whole columns dealt to the XCDs in turn 11 x 20 tiles took two rounds on four of them.)
__device__ __forceinline__ bool tiles_place(int tiles, int rows, int cols, int xcd, int j, int& row, int& col) {
    const int per = tiles >> 3, more = tiles & 7;
    if (j >= per + (xcd < more)) return false;
    const int id = xcd * per + min(xcd, more) + j, band = id / (8 * cols), at = id - band * 8 * cols, high = min(8, rows - 8 * band);
    col = at / high;
    row = 8 * band + at % high;
    return true;
}

constexpr int kTileWaves = 4;
constexpr int kTileBlocks = 4;                         // packed blocks of 64 rows of w a tile: 256 rows, a block a wave
constexpr int kStageK = 64;
constexpr int kRing = 4;                               // stages of 64 k in LDS and in registers
enum { EPI_PLAIN = 0, EPI_SWIGLU = 1, EPI_ADD = 2, EPI_ROWS = 3, EPI_ROWS_GATED = 4,   // (sorted rows of experts, moe_packed.hip)
       EPI_RELU2 = 5, EPI_XIELU = 6 };                              // activations with what activation.h takes (TileEnd: act_a, act_b)

constexpr int tiles_lds_bytes(int tm) { return kRing * tm * 16 * kStageK * 2; }

// silu(gate) * up, or, with limit >= 0, g = min(gate, limit), u = up within -limit .. limit, g * sigmoid(1.702 g) * (u + 1).  (Selects
// and no branch, of which there would be one a value.)
__device__ __forceinline__ float tiles_gated(float gate, float up, float limit) {
    const bool bounded = limit >= 0.f;
    const float g = bounded ? fminf(gate, limit) : gate, u = bounded ? fminf(fmaxf(up, -limit), limit) + 1.0f : up;
    return g / (1.0f + __expf((bounded ? -1.702f : -1.0f) * g)) * u;
}

// the same for experts, whose other kernels take the exact exponential
__device__ __forceinline__ float tiles_rows_gated(float gate, float up, float limit) {
    const bool bounded = limit >= 0.f;
    const float g = bounded ? fminf(gate, limit) : gate, u = bounded ? fminf(fmaxf(up, -limit), limit) + 1.0f : up;
    return g / (1.0f + expf((bounded ? -1.702f : -1.0f) * g)) * u;
}

template <int N> __device__ __forceinline__ void tiles_wait_loads() {
    static_assert(N < 64, "the counter has six bits");
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

// The products of one tile: acc[token tile][strip] += 16 TM rows of activations . a wave's 64 rows of w over `stages` stages of 64 k.  w_base:
// the wave's packed block at the first stage; a_base + a_off[i]: where lane l finds octet (l & 7) ^ ((row >> 1) & 7) of row
// 8 (wave TM / 2 + i) + (l >> 3) of the tile at the first stage (tiles_a_row), offsets below 2^31.
template <int TM> __device__ __forceinline__ int tiles_a_row(int i) { return 8 * ((int)(threadIdx.x / kWave) * (TM / 2) + i) + ((threadIdx.x & (kWave - 1)) >> 3); }

template <int TM>
__device__ __forceinline__ void tile_products(unsigned char* lds, f32x4_t (&acc)[TM][4], const unsigned char* w_base, const unsigned char* a_base,
                                              const unsigned (&a_off)[TM / 2], int stages) {
#ifdef __HIP_DEVICE_COMPILE__
    constexpr int kBuf = TM * 16 * kStageK * 2;
    constexpr int kCopies = TM / 2;                          // copies of 8 rows of activations, a wave and stage
    constexpr int kLoads = 8 + kCopies;                      // and 8 operands of w
    constexpr int kUnits = 2 * TM;                           // of a stage: 32 k of 16 tokens against the wave's 64 rows, four products
    constexpr int kFrags = kUnits % 8 == 0 ? 8 : TM == 14 ? 7 : TM;
    constexpr int kAhead = TM == 4 ? 3 : TM == 6 ? 4 : TM == 8 ? 4 : 6;
    constexpr int kLag = kAhead > 4 ? 2 : 1, kMeet = kUnits - kAhead + kLag;
    constexpr int kBefore = kLoads * kMeet / kUnits;         // loads of a stage that are asked for before the barrier ...
    constexpr int kWait = kLoads + kBefore;                  // ... and the whole stage before: what may still be on its way then
    static_assert(kWait > kLoads && kWait < 64, "a whole stage stays on its way, in a counter of six bits");
    static_assert(TM % 2 == 0 && kUnits % kFrags == 0 && kAhead < kFrags && 2 * kLag <= kAhead, "a tile's schedule");

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i16 = lane & 15, g = lane >> 4;
    // The weights' pointer is hidden from the compiler: it could otherwise tell that nothing writes what it points to, and move
    // loads past the barriers.
    asm volatile("" : "+s"(w_base));
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)w_base, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a_base, 0, 0x7fffffff, 0x00020000);
    const unsigned w_off = lane * 16;
    int a_read[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) a_read[j] = i16 * 128 + (((4 * j + g) ^ ((i16 >> 1) & 7)) * 16);

#pragma unroll
    for (int tt = 0; tt < TM; ++tt)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) acc[tt][rt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    u32x4_t w[kRing][2][4];
    u32x4_t f[kFrags];
    // load l of a stage into a place of the ring.  Beyond the part's last stage the offset lies past the buffer's end: such loads
    // bring zeros and read nothing.
    auto load = [&](int slot, int l, int stage, unsigned past) {
        const int na = kCopies * (l + 1) / kLoads;
        if (na > kCopies * l / kLoads) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc,
                (__attribute__((address_space(3))) void*)(lds + slot * kBuf + (wave * kCopies + na - 1) * 1024), 16, a_off[na - 1] | past, stage * 128, 0, 0);
        } else {
            const int i = l - na;
            w[slot][i >> 2][i & 3] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (w_off | past) + (i & 3) * 1024, stage * 8192 + (i >> 2) * 4096, 0);
        }
    };
    auto read_a = [&](int slot, int unit) {
        f[unit % kFrags] = *reinterpret_cast<const u32x4_t*>(lds + slot * kBuf + a_read[unit / TM] + (unit % TM) * 2048);
    };
    auto meet = [&]() {
        SB();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        SB();
    };
    auto past_end = [&](int stage) { return stage < stages ? 0u : 0x80000000u; };
    auto stage_body = [&](auto place, int s) {
        constexpr int b = decltype(place)::value;
        const unsigned past = past_end(s + 3);
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            if (u == kMeet) {
                // this stage's fragments are all here (its buffer is the next to be written), and this wave's copies of the next
                // stage too: loads come back in the order in which they were asked for (the compiler's own waits for w, which count
                // copies and loads alike, rest on that too), so all but the kWait youngest are here.  (A wait that counted
                // copies alone left no stage on its way: [2,048, 8,192], 65 rows in eight parts 19.2 us, 16.5 now; [4,096, 14,336] 32.3
                // and 27.6; in one part a fifth; from 3,000 rows on level.)
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                tiles_wait_loads<kWait>();
                meet();
            }
            if (u + kAhead < kUnits) read_a(b, u + kAhead);
            else if (u >= kMeet) {
#pragma unroll
                for (int r = 0; r < kAhead; ++r)             // two a unit until they are kAhead ahead again
                    if ((r < 2 * kLag ? r / 2 : r - kLag) == u - kMeet) read_a((b + 1) & 3, r);
            }
            SB();
            const int ks = u / TM, tt = u % TM;
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                acc[tt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[b][ks][rt]),
                                                                      __builtin_bit_cast(bf16x8_t, f[u % kFrags]), acc[tt][rt], 0, 0, 0);
                SB();
                if (rt == 1) {
#pragma unroll
                    for (int l = kLoads * u / kUnits; l < kLoads * (u + 1) / kUnits; ++l) load((b + 3) & 3, l, s + 3, past);
                    SB();
                }
            }
        }
    };
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int l = 0; l < kLoads; ++l) load(p, l, p, past_end(p));
    SB();
    tiles_wait_loads<2 * kLoads>();
    meet();
#pragma unroll
    for (int u = 0; u < kAhead; ++u) read_a(0, u);
    SB();
    int s = 0;
    do {                                                     // (whole rounds of the ring: the stages past the last add zeros)
        stage_body(std::integral_constant<int, 0>{}, s);
        stage_body(std::integral_constant<int, 1>{}, s + 1);
        stage_body(std::integral_constant<int, 2>{}, s + 2);
        stage_body(std::integral_constant<int, 3>{}, s + 3);
        s += 4;
    } while (s < stages);
    tiles_wait_loads<0>();                                   // copies still on their way into LDS
    __syncthreads();

#endif
}

// What an epilogue needs of its tile.  out: rows ldo apart, width values each; token rows m0 .. m_end - 1; the wave's packed block of rows nb of n_row_blocks.
struct TileEnd {
    int m0, m_end, N, ldo, nb, n_row_blocks;
    const float* bias;
    float limit;
    // of experts: the epilogue (0 as they are, 1 squares of what is above 0, 2 and 3 gated, 3 bounded), a factor, a weight for each row
    int act;
    float scale;
    const float* row_weight;
    const int* order;
    float act_a, act_b;
};

template <int TM, int EPI, typename TO>
__device__ __forceinline__ void tile_store(unsigned char* lds, f32x4_t (&acc)[TM][4], TO* __restrict__ out, const TileEnd& at) {
#ifdef __HIP_DEVICE_COMPILE__
    constexpr int BM = TM * 16, kBuf = BM * kStageK * 2;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i16 = lane & 15, g = lane >> 4, nb = at.nb, N = at.N, ldo = at.ldo, m0 = at.m0;
    float limit = at.limit;
    if (nb >= at.n_row_blocks) return;
    // Results go through the wave's own quarter of LDS, so that rows of 64 to 256 bytes are stored 16 bytes a lane: tokens a pass,
    // 16-byte pieces of a row, tokens a store.
    constexpr bool kGated = EPI == EPI_SWIGLU || EPI == EPI_ROWS_GATED;
    constexpr int kVals = kGated ? 32 : 64, kEach = 16 / (int)sizeof(TO), kPieces = kVals / kEach;
    constexpr int kRegion = kRing * kBuf / kTileWaves, kRowBytes = kPieces * 16;
    constexpr int kPass = kRegion / kRowBytes < BM ? kRegion / kRowBytes : BM, kTokens = kWave / kPieces;
    static_assert(kPass % 16 == 0 && BM % kPass == 0, "whole token tiles a pass");
    unsigned char* mine = lds + wave * kRegion;
    const int width = kGated ? N / 2 : N, col0 = kVals * nb;
    const bool wide = (ldo % kEach) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    if (kGated) asm("" : "+v"(limit));           // (not known to be the same in all lanes: selects instead of branches)
    f32x4_t more[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = 64 * nb + 16 * rt + 4 * g + e;
            more[rt][e] = EPI == EPI_PLAIN && at.bias && n < N ? at.bias[n] : 0.f;
        }
    auto put = [&](int t, int value, f32x4_t y) {            // values value .. value + 3 of token t of the pass
        const int piece = value / kEach;
        unsigned char* at = mine + t * kRowBytes + ((piece ^ (t & (kPieces - 1))) * 16);
        if (sizeof(TO) == 4) *reinterpret_cast<f32x4_t*>(at) = y;
        else *reinterpret_cast<uint2*>(at + (value & 4) * 2) = make_uint2(tiles_pack_bf16(y[0], y[1]), tiles_pack_bf16(y[2], y[3]));
    };
#pragma unroll
    for (int p0 = 0; p0 < BM; p0 += kPass) {
#pragma unroll
        for (int tt = p0 / 16; tt < (p0 + kPass) / 16; ++tt) {
            const int t = 16 * tt - p0 + i16;
            // The sums leave the accumulation registers by a product with one, hidden and made anew for each 16 tokens: else the
            // compiler keeps some of them in ordinary registers throughout and copies them in the loop, or spills.
            float one = 1.0f;
            asm volatile("" : "+s"(one));
            if (EPI == EPI_SWIGLU) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    f32x4_t y = acc[tt][2 * i] * one, up = acc[tt][2 * i + 1] * one;
                    asm volatile("" : "+v"(y), "+v"(up));
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] = tiles_gated(y[e], up[e], limit);
                    SB();
                    put(t, 16 * i + 4 * g, y);
                }
            } else if (EPI == EPI_ROWS_GATED) {              // gate and up in turn: a lane's four sums are two of the result's columns
                const float rw = at.row_weight ? at.row_weight[at.order[min(m0 + 16 * tt + i16, at.m_end - 1)]] : 1.0f;
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) {
                    f32x4_t y = acc[tt][rt] * one;
                    asm volatile("" : "+v"(y));
                    const float lo = tiles_rows_gated(y[0] * rw, y[1] * rw, limit) * at.scale, hi = tiles_rows_gated(y[2] * rw, y[3] * rw, limit) * at.scale;
                    const int value = 8 * rt + 2 * g, piece = value / kEach;
                    unsigned char* to = mine + t * kRowBytes + ((piece ^ (t & (kPieces - 1))) * 16) + value % kEach * (int)sizeof(TO);
                    if (sizeof(TO) == 4) *reinterpret_cast<float2*>(to) = make_float2(lo, hi);
                    else *reinterpret_cast<uint32_t*>(to) = tiles_pack_bf16(lo, hi);
                    SB();
                }
            } else {
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) {
                    f32x4_t y = acc[tt][rt] * one;
                    if (EPI == EPI_ROWS) {
                        asm volatile("" : "+v"(y));
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = fmaxf(y[e], 0.f);
                            y[e] = (at.act == 1 ? v * v : y[e]) * at.scale;
                        }
                    }
                    if (EPI == EPI_RELU2 || EPI == EPI_XIELU) {
                        asm volatile("" : "+v"(y));
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[e] = activate(y[e], EPI == EPI_RELU2 ? ACT_RELU2 : ACT_XIELU, at.act_a, at.act_b);
                    }
                    if (EPI == EPI_PLAIN && at.bias) y += more[rt];
                    put(t, 16 * rt + 4 * g, y);
                }
            }
            SB();
        }
        asm volatile("" ::: "memory");
        const int piece = lane % kPieces, col = col0 + kEach * piece;
#pragma unroll 8
        for (int it = 0; it < kPass / kTokens; ++it) {
            const int t = kTokens * it + lane / kPieces, token = m0 + p0 + t;
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(mine + t * kRowBytes + ((piece ^ (t & (kPieces - 1))) * 16));
            if (token >= at.m_end) continue;
            TO* o = out + (size_t)token * ldo + col;
            if (wide && col + kEach <= width) {
                if (EPI == EPI_ADD) {
                    const f32x4_t sum = *reinterpret_cast<const f32x4_t*>(o) + __builtin_bit_cast(f32x4_t, v);
                    __builtin_nontemporal_store(sum, reinterpret_cast<f32x4_t*>(o));
                } else {
                    __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(o));
                }
            } else {
#pragma unroll
                for (int e = 0; e < kEach; ++e) {
                    if (col + e >= width) continue;
                    if (sizeof(TO) == 4) {
                        const float y = __uint_as_float(v[e]);
                        store_f32(o + e, EPI == EPI_ADD ? y + load_f32(o + e) : y);
                    } else {
                        o[e] = (TO)(v[e / 2] >> (16 * (e & 1)));
                    }
                }
            }
        }
        asm volatile("" ::: "memory");
    }
#endif
}

// One tile: 16 TM tokens by 256 rows of w, stages [stage_begin, stage_end) of k.  out: EPI_SWIGLU [M][N / 2], else [M][N], rows ldo apart.  limit: of the
// gated form, or an activation's first number.
template <int TM, int EPI, typename TO>
__device__ __forceinline__ void tile_body(
        unsigned char* lds, TO* __restrict__ out, const bf16_t* __restrict__ a, int lda, const unsigned char* __restrict__ wp,
        const float* __restrict__ bias, int M, int N, int K, int ldo, int n_row_blocks, int m_tile, int n_tile, int stage_begin,
        int stage_end, float limit, float act_b) {
    const int m0 = m_tile * TM * 16, nb = n_tile * kTileBlocks + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const unsigned char* w_base = wp + ((size_t)min(nb, n_row_blocks - 1) * (K / 32) + 2 * stage_begin) * 4096;
    const unsigned char* a_base = reinterpret_cast<const unsigned char*>(a + (size_t)m0 * lda + (size_t)stage_begin * kStageK);
    unsigned a_off[TM / 2];
#pragma unroll
    for (int i = 0; i < TM / 2; ++i) {
        const int row = tiles_a_row<TM>(i);
        a_off[i] = (unsigned)min(row, M - 1 - m0) * (unsigned)(lda * 2) + 16 * ((threadIdx.x & 7) ^ ((row >> 1) & 7));
    }
    f32x4_t acc[TM][4];
    tile_products<TM>(lds, acc, w_base, a_base, a_off, stage_end - stage_begin);
    TileEnd at{};
    at.m0 = m0, at.m_end = M, at.N = N, at.ldo = ldo, at.nb = nb, at.n_row_blocks = n_row_blocks, at.bias = bias, at.limit = limit, at.act_a = limit, at.act_b = act_b;
    tile_store<TM, EPI, TO>(lds, acc, out, at);
}

// A launch, as the entry points hand it to the file that holds its kernels.  rows, rows_last: units of 16 tokens a tile; row tiles
// n_full and up come in tiles of rows_last (half of rows) where that is not 0.
struct TilesCall {
    void* out;
    const void* a;
    const void* wp;
    const float* bias;
    int lda, M, N, K, ldo, parts, rows, rows_last, n_full;
    long long part_stride;
    float limit, act_b;
    hipStream_t stream;
};
// (one file each, so that they are compiled side by side)
int tiles_plain_f32(const TilesCall& c);
int tiles_plain_bf16(const TilesCall& c);
int tiles_add_f32(const TilesCall& c);
int tiles_gated_f32(const TilesCall& c);
int tiles_gated_bf16(const TilesCall& c);
int tiles_relu2_bf16(const TilesCall& c);
int tiles_xielu_bf16(const TilesCall& c);

// Blocks 0 .. blocks_full - 1 take tiles of 16 TM tokens over the first n_full row tiles, the blocks after them tiles of 16 TS tokens
// over the remaining row tiles (TS = 0: there are none).
template <int TM, int TS, int EPI, typename TO>
__global__ __launch_bounds__(kTileWaves * kWave, 1) void gemm_tiles_kernel(
        TO* __restrict__ out, const bf16_t* __restrict__ a, int lda, const unsigned char* __restrict__ wp,
        const float* __restrict__ bias, int M, int N, int K, int ldo, size_t part_stride, int n_row_blocks,
        int m_full, int m_last, int n_full, int n_tiles, int blocks_full, int parts, float limit, float act_b) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char tiles_lds[];
    const int stages = K / kStageK;
    const bool full = TS == 0 || (int)blockIdx.x < blocks_full;
    const int b = full ? blockIdx.x : blockIdx.x - blocks_full;              // (blocks_full is a multiple of 8)
    const int m_tiles = full ? m_full : m_last, across = full ? n_full : n_tiles - n_full;
    int m_tile, u;
    if (!tiles_place(m_tiles * across * parts, m_tiles, across * parts, b & 7, b >> 3, m_tile, u)) return;
    const int part = u / across, n_tile = (full ? 0 : n_full) + u % across;
    // the parts divide the stages evenly: part p takes [stages p / parts, stages (p + 1) / parts), none is empty
    // when there are at least as many stages as parts
    const int s0 = (int)((long long)stages * part / parts), s1 = (int)((long long)stages * (part + 1) / parts);
    TO* dst = out + (size_t)part * part_stride;
    if (full) tile_body<TM, EPI, TO>(tiles_lds, dst, a, lda, wp, bias, M, N, K, ldo, n_row_blocks, m_tile, n_tile, s0, s1, limit, act_b);
    else if (TS > 0) tile_body<(TS > 0 ? TS : 4), EPI, TO>(tiles_lds, dst, a, lda, wp, bias, M, N, K, ldo, n_row_blocks, m_tile, n_tile, s0, s1, limit, act_b);
}

template <int TM, int TS, int EPI, typename TO>
int launch_tile_kernel(const TilesCall& c) {
    const int n_row_blocks = (c.N + 63) / 64, n_tiles = (n_row_blocks + kTileBlocks - 1) / kTileBlocks;
    const int n_full = TS > 0 ? c.n_full : n_tiles, m_full = (c.M + 16 * TM - 1) / (16 * TM), m_last = TS > 0 ? (c.M + 16 * TS - 1) / (16 * TS) : 0;
    const long long full = ((long long)m_full * n_full * c.parts + 7) / 8 * 8, last = ((long long)m_last * (n_tiles - n_full) * c.parts + 7) / 8 * 8;
    if (full + last > 1 << 26) return LLOGOS_UNSUPPORTED;
    constexpr int smem = tiles_lds_bytes(TM);
    static std::atomic<uint64_t> asked{0};
    const int code = allow_dynamic_lds((const void*)gemm_tiles_kernel<TM, TS, EPI, TO>, smem, asked);
    if (code != 0) return code;
    gemm_tiles_kernel<TM, TS, EPI, TO><<<(unsigned)(full + last), kTileWaves * kWave, smem, c.stream>>>(
        (TO*)c.out, (const bf16_t*)c.a, c.lda, (const unsigned char*)c.wp, c.bias, c.M, c.N, c.K, c.ldo, (size_t)c.part_stride, n_row_blocks,
        m_full, m_last, n_full, n_tiles, (int)full, c.parts, c.limit, c.act_b);
    return LLOGOS_LAUNCH_CHECK();
}

template <int EPI, typename TO>
int launch_tiles(const TilesCall& c) {
    switch (c.rows) {
        case 4: return launch_tile_kernel<4, 0, EPI, TO>(c);
        case 6: return launch_tile_kernel<6, 0, EPI, TO>(c);
        case 8: return launch_tile_kernel<8, 0, EPI, TO>(c);
        case 10: return launch_tile_kernel<10, 0, EPI, TO>(c);
        case 12: return launch_tile_kernel<12, 0, EPI, TO>(c);
        case 14: return launch_tile_kernel<14, 0, EPI, TO>(c);
        case 16: return c.rows_last ? launch_tile_kernel<16, 8, EPI, TO>(c) : launch_tile_kernel<16, 0, EPI, TO>(c);
    }
    return LLOGOS_BAD_ARGUMENT;
}
