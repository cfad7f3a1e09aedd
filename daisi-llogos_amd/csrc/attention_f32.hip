// Attention of the float32 engine over the paged cache on the matrix cores' 32-bit instruction
// (v_mfma_f32_16x16x4f32: a chain of four fused multiply-adds, nothing is rounded to fewer bits),
// for heads of 64 and 128 dimensions; a window and sinks as in the kernel for any shape.
//
// A block takes 16 query rows of one sequence and kv head: rows are (token, head of the group)
// pairs in order, so that the heads that share keys share a tile whatever the group's size.  Its
// waves take the sequence's pages in turn.  A page is worked on by itself: scores of its 64 keys,
// their maximum and sum, the weighted sum of its values from zero; the pages' results go through
// LDS and are added in ascending order with the running maximum.  The order of every addition so
// depends on the query's position alone, not on how many waves share the pages, on how the tokens
// were cut into steps or on what else is in the batch: single tokens and prompts run this kernel
// with the same bits.  (A page of which a row sees no key leaves the row as it was: factors 1 and
// 0.)  A key whose weight is 0, unseen or underflowed, counts for nothing whatever its value is.
//
// Bound by the latency of a page's loads in single-token steps and by the matrix cores in prompts
// (a page of 16 rows of 64 dimensions: 128 instructions, 4,096 clocks).  The kernel for any shape
// gave a block to every (token, head), whose threads walk keys and values with scalar loads.
// Measured (us, before -> now): heads of 64, 32 to 8 kv heads, prompts of 515 and 190 tokens 1,019 -> 47, one of 2,048
// tokens 14,731 -> 288; single tokens behind 515 and 190: 158 -> 10, behind 8,192: 2,625 -> 38.  Heads of 128: 1,496 -> 90,
// 19,143 -> 536, 180 -> 15, 2,721 -> 47.
// Behind only where a step's longest context has fewer than some 16 tokens, since a page is worked on whole: one token of heads
// of 64 by itself 4.9 -> 6.6, of 128 5.9 -> 10.6, a prompt of 16 11.2 -> 11.8 (the other kernel adds in another order, so
// serving those with it would cost the bits that a token has in common with itself in a longer step).
//
// Single tokens of few sequences leave most of the chip without a block, and sixteen pages on one compute unit are four for each of
// its matrix units, 7 us; their pages go to several blocks (attn_f32_shared_kernel, attn_f32_pages_kernel), 2 sequences of 8 kv heads
// behind 1,000 tokens 19.5 -> 11.2.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8), aligned(16)));

// One page of a tile of 16 rows by itself: the maximum m and the sum l of this lane's row and its weighted sum of values, o[d][r] of dimension
// 16 d + 4 g + r.  t0: the page's first token; last: the tile's latest position.
template <int HD>
__device__ __forceinline__ void attn_f32_page(const float* __restrict__ kp, const float* __restrict__ vp, const f32x8 (&qv)[HD / 32], int pos, int last,
                                              int t0, float scale, int window, int sinks, float& m, float& l, f32x4 (&o)[HD / 16]) {
    constexpr int DB = HD / 16;
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    // S^T = K . Q^T: block rb of four tokens gives lane (i, g) the scores of row i with tokens 16 g + 4 rb .. + 3
    f32x4 s[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
        f32x8 kv[HD / 32];
#pragma unroll
        for (int d = 0; d < HD / 32; ++d)
            kv[d] = *reinterpret_cast<const f32x8*>(kp + ((rb * (HD / 8) + 4 * d + g) * 16 + i) * 8);
        s[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < HD / 32; ++d)
#pragma unroll
            for (int e = 0; e < 8; ++e) s[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[d][e], qv[d][e], s[rb], 0, 0, 0);
    }
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = t0 + 16 * g + 4 * rb + r;
            s[rb][r] = key_visible(pos, t, window, sinks) ? s[rb][r] * scale : -INFINITY;
            m = fmaxf(m, s[rb][r]);
        }
    m = fmaxf(m, __shfl_xor(m, 16, kWave));
    m = fmaxf(m, __shfl_xor(m, 32, kWave));
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[rb][r] = m == -INFINITY ? 0.f : expf(s[rb][r] - m);
            l += s[rb][r];
        }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    // O^T = V^T . P^T; values behind the tile's latest position were never written
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int d = 0; d < DB; ++d) {
            f32x8 vv = *reinterpret_cast<const f32x8*>(vp + (((d * 2 + h) * 4 + g) * 16 + i) * 8);
            if (t0 + kPageTokens - 1 > last) {
#pragma unroll
                for (int e = 0; e < 8; ++e) if (t0 + 16 * g + 8 * h + e > last) vv[e] = 0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[e], s[2 * h + (e >> 2)][e & 3], o[d], 0, 0, 0);
        }
    // A weight of 0 (a key that the row does not see, or one whose weight underflows) must not meet a value that is no
    // number, and every such meeting leaves a sum that is no number: then the page is added token by token without
    // them, in the instruction's order (slot g of step j holds token 16 g + j), so that rows that do not see the value
    // keep their bits.
    bool odd = false;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int c = 0; c < 4; ++c) odd |= !isfinite(o[d][c]);
    if (__any(odd)) {
#pragma unroll
        for (int d = 0; d < DB; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 16; ++j)
#pragma unroll 1
            for (int u = 0; u < 4; ++u) {
                const float p = __shfl(s[j >> 2][j & 3], 16 * u + i, kWave);
                if (p != 0.f) {
#pragma unroll
                    for (int d = 0; d < DB; ++d)
#pragma unroll
                        for (int c = 0; c < 4; ++c) o[d][c] = fmaf(p, vp[page_value_offset(16 * u + j, 16 * d + 4 * g + c)], o[d][c]);
                }
            }
    }
}

// cu: token offsets of the sequences [batch + 1]; null: every sequence brings one token.  tok_seq: row of the page table a
// token's sequence has; null: the sequences' own order.  A sequence's tokens may come in any order of positions.
template <int HD, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void attn_f32_kernel(
        float* __restrict__ out, const float* __restrict__ q, int q_stride, const float* __restrict__ k_pool,
        const float* __restrict__ v_pool, PagedKV cache, const int* __restrict__ cu, int batch,
        const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, int n_heads, int group, float scale, int window, int sinks) {
    constexpr int DB = HD / 16, OWN = (DB + WAVES - 1) / WAVES;
    __shared__ f32x4 sums[WAVES][DB][64];
    __shared__ float tops[WAVES][16], dens[WAVES][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
    const int kvh = blockIdx.y;

    // which sequence this tile of rows belongs to; the tiles of late tokens, which have most pages, go first
    int seq = 0, first = 0, tokens = 1, tile = gridDim.x - 1 - blockIdx.x;
    if (cu) {
        // (the lanes look at 64 sequences side by side: one after the other each costs a round trip to the cache)
        for (int s0 = 0;; s0 += kWave) {
            if (s0 >= batch) return;                             // (the grid has up to a tile a sequence more than there are)
            const int lo = cu[min(s0 + lane, batch)], hi = cu[min(s0 + lane + 1, batch)];
            const int tiles = ((hi - lo) * group + 15) / 16;
            int upto = tiles;                                    // tiles of this sequence and the ones in front of it
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) { const int v = __shfl_up(upto, o, kWave); if (lane >= o) upto += v; }
            const unsigned long long mine = __ballot(tile < upto);
            if (mine) {
                const int at = __ffsll(mine) - 1;
                seq = s0 + at;
                first = __builtin_amdgcn_readlane(lo, at);
                tokens = __builtin_amdgcn_readlane(hi, at) - first;
                tile -= __builtin_amdgcn_readlane(upto - tiles, at);
                break;
            }
            tile -= __builtin_amdgcn_readlane(upto, kWave - 1);
        }
    } else {
        const int tiles = (group + 15) / 16;
        seq = tile / tiles;
        tile -= seq * tiles;
        first = seq;
    }
    const int rows = tokens * group, row = tile * 16 + i;        // this lane's query row (columns of the products)
    const bool real = row < rows;
    const int tok = first + min(row, rows - 1) / group, head = kvh * group + min(row, rows - 1) % group;
    const int pos = real ? tok_pos[tok] : -1;
    int last = pos, early = real ? pos : 0x7fffffff;             // the tile's latest position and its earliest
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) { last = max(last, __shfl_xor(last, o, kWave)); early = min(early, __shfl_xor(early, o, kWave)); }
    last = __builtin_amdgcn_readfirstlane(last);                // (the same in every lane)
    early = __builtin_amdgcn_readfirstlane(early);
    if (tok_seq) seq = tok_seq[first];

    f32x8 qv[HD / 32];
#pragma unroll
    for (int d = 0; d < HD / 32; ++d)
        qv[d] = *reinterpret_cast<const f32x8*>(q + (size_t)tok * q_stride + (size_t)head * HD + 32 * d + 8 * g);

    f32x4 acc[OWN];
    float top = -INFINITY, den = 0.f;
#pragma unroll
    for (int o = 0; o < OWN; ++o) acc[o] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int pages = last / kPageTokens + 1;
    for (int p0 = 0; p0 < pages; p0 += WAVES) {                  // the same trips for every wave: the barriers match
        // pages that no row of the tile sees may have been given back: nothing of them is read
        if (window > 0 && p0 * kPageTokens >= sinks && (p0 + WAVES) * kPageTokens - 1 <= early - window) continue;
        const int page = p0 + wave, t0 = page * kPageTokens;
        const bool seen = page < pages && !(window > 0 && t0 >= sinks && t0 + kPageTokens - 1 <= early - window);
        float m = -INFINITY, l = 0.f;
        f32x4 o[DB];
#pragma unroll
        for (int d = 0; d < DB; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (seen) {
            const size_t base = paged_base(cache, seq, kvh, t0);
            const float* kp = k_pool + base;
            const float* vp = v_pool + base;
            attn_f32_page<HD>(kp, vp, qv, pos, last, t0, scale, window, sinks, m, l, o);
        }
#pragma unroll
        for (int d = 0; d < DB; ++d) sums[wave][d][lane] = o[d];
        if (g == 0) { tops[wave][i] = m; dens[wave][i] = l; }
        __syncthreads();
        const int here = min(WAVES, pages - p0);
        for (int j = 0; j < here; ++j) {
            const float mj = tops[j][i];
            const float high = fmaxf(top, mj);
            const float keep = top == -INFINITY ? 0.f : expf(top - high), add = mj == -INFINITY ? 0.f : expf(mj - high);
#pragma unroll
            for (int w = 0; w < OWN; ++w) {
                const int d = wave + w * WAVES;
                if (d < DB) {
                    const f32x4 v = sums[j][d][lane];
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[w][r] = fmaf(add == 0.f ? 0.f : v[r], add, (keep == 0.f ? 0.f : acc[w][r]) * keep);
                }
            }
            den = fmaf(dens[j][i], add, den * keep);
            top = high;
        }
        __syncthreads();
    }
    const float inv = den > 0.f ? 1.0f / den : 0.f;
    if (!real) return;
#pragma unroll
    for (int w = 0; w < OWN; ++w) {
        const int d = wave + w * WAVES;
        if (d < DB) {
            f32x4 v = acc[w];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= inv;
            *reinterpret_cast<f32x4*>(out + ((size_t)tok * n_heads + head) * HD + 16 * d + 4 * g) = v;
        }
    }
}

// floats of a page's share: its rows' sums of HD dimensions, then a row's maximum and sum of weights, to whole 16 bytes
__host__ __device__ constexpr int attn_f32_share(int rows, int hd) { return (rows * (hd + 2) + 3) & ~3; }

// A single-token step's pages side by side: a block of one wave takes every gridDim.z-th page of a tile and leaves the page's sums, maximum and sum of
// weights in `shares` [tile][kv head][page of `pages`][rows x HD sums, rows x (maximum, sum)]; attn_f32_pages_merge adds them.  Bound by the
// latency of a page's loads and by the launch of the second kernel: heads of 64, 8 kv heads, one sequence behind 2,000 tokens 35.3 -> 14.8.
template <int HD>
__global__ __launch_bounds__(64) void attn_f32_pages_kernel(
        float* __restrict__ shares, const float* __restrict__ q, int q_stride, const float* __restrict__ k_pool, const float* __restrict__ v_pool,
        PagedKV cache, int pages, const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, int group, float scale, int window, int sinks) {
    constexpr int DB = HD / 16;
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4, kvh = blockIdx.y;
    const int tiles = (group + 15) / 16, tok = blockIdx.x / tiles, first = 16 * (blockIdx.x - tok * tiles), rows = min(16, group);
    const bool real = first + i < group;
    const int head = kvh * group + min(first + i, group - 1), at = __builtin_amdgcn_readfirstlane(tok_pos[tok]), pos = real ? at : -1;
    const int seq = tok_seq ? tok_seq[tok] : tok, n_pages = min(at / kPageTokens + 1, pages);
    if ((int)blockIdx.z >= n_pages) return;
    f32x8 qv[HD / 32];
#pragma unroll
    for (int d = 0; d < HD / 32; ++d)
        qv[d] = *reinterpret_cast<const f32x8*>(q + (size_t)tok * q_stride + (size_t)head * HD + 32 * d + 8 * g);
    float* mine = shares + ((size_t)blockIdx.x * gridDim.y + kvh) * pages * attn_f32_share(rows, HD);
    for (int page = blockIdx.z; page < n_pages; page += gridDim.z) {
        const int t0 = page * kPageTokens;
        if (window > 0 && t0 >= sinks && t0 + kPageTokens - 1 <= at - window) continue;      // (the merge skips it too)
        float m = -INFINITY, l = 0.f;
        f32x4 o[DB];
#pragma unroll
        for (int d = 0; d < DB; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
        const size_t base = paged_base(cache, seq, kvh, t0);
        attn_f32_page<HD>(k_pool + base, v_pool + base, qv, pos, at, t0, scale, window, sinks, m, l, o);
        float* share = mine + (size_t)page * attn_f32_share(rows, HD);
        if (real) {
#pragma unroll
            for (int d = 0; d < DB; ++d) *reinterpret_cast<f32x4*>(share + i * HD + 16 * d + 4 * g) = o[d];
            if (g == 0) *reinterpret_cast<float2*>(share + rows * HD + 2 * i) = make_float2(m, l);
        }
    }
}

// The shares in ascending order of the pages, by the arithmetic of attn_f32_kernel: a thread has four dimensions of a row.  Bound by latency: eight
// pages' shares are asked for at a time.
template <int HD>
__global__ void attn_f32_pages_merge(float* __restrict__ out, const float* __restrict__ shares, int pages, const int* __restrict__ tok_pos,
                                     int n_heads, int group, int window, int sinks) {
    constexpr int kAt = 8;
    const int kvh = blockIdx.y, rows = min(16, group), i = threadIdx.x / (HD / 4), c = 4 * (threadIdx.x % (HD / 4));
    const int tiles = (group + 15) / 16, tok = blockIdx.x / tiles, first = 16 * (blockIdx.x - tok * tiles);
    if (first + i >= group) return;
    const int pos = tok_pos[tok], n_pages = min(pos / kPageTokens + 1, pages);
    const float* mine = shares + ((size_t)blockIdx.x * gridDim.y + kvh) * pages * attn_f32_share(rows, HD);
    float top = -INFINITY, den = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int p0 = 0; p0 < n_pages; p0 += kAt) {
        f32x4 v[kAt];
        float2 ml[kAt];
#pragma unroll
        for (int j = 0; j < kAt; ++j) {
            const int t0 = (p0 + j) * kPageTokens;
            const bool there = p0 + j < n_pages && !(window > 0 && t0 >= sinks && t0 + kPageTokens - 1 <= pos - window);
            const float* share = mine + (size_t)(p0 + j) * attn_f32_share(rows, HD);
            v[j] = there ? *reinterpret_cast<const f32x4*>(share + i * HD + c) : f32x4{0.f, 0.f, 0.f, 0.f};
            ml[j] = there ? *reinterpret_cast<const float2*>(share + rows * HD + 2 * i) : make_float2(-INFINITY, 0.f);
        }
#pragma unroll
        for (int j = 0; j < kAt; ++j) {
            const float mj = ml[j].x, high = fmaxf(top, mj);
            const float keep = top == -INFINITY ? 0.f : expf(top - high), add = mj == -INFINITY ? 0.f : expf(mj - high);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = fmaf(add == 0.f ? 0.f : v[j][r], add, (keep == 0.f ? 0.f : acc[r]) * keep);
            den = fmaf(ml[j].y, add, den * keep);
            top = high;
        }
    }
    const float inv = den > 0.f ? 1.0f / den : 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] *= inv;
    *reinterpret_cast<f32x4*>(out + ((size_t)tok * n_heads + kvh * group + first + i) * HD + c) = acc;
}

// A page's sums as two pairs that pass the L2 of the XCD, which the block that adds them may not share.
__device__ __forceinline__ void share_store(float* p, float x, float y) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, make_float2(x, y)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 share_load(const float* p) {
    return __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// The same for tables of up to kSharedPages pages, in one kernel: blocks of four waves, a page a wave.  Up to four pages are one block's, which adds
// them through LDS.  Beyond, a block writes its pages' shares past the L2, waits until they have arrived and takes a ticket, and the one with the
// last ticket reads them past its own and adds them in the same order (nobody waits for another block; the counter is back at zero then; what that
// rests on stands with attn_decode_kernel's tickets).  8 kv heads of 64, one sequence: 7.7 -> 6.6 us behind 40 tokens, 12.1 -> 10.1 behind 500.
constexpr int kSharedPages = 16;

template <int HD>
__global__ __launch_bounds__(256) void attn_f32_shared_kernel(
        float* __restrict__ out, float* shares, unsigned* tickets, const float* __restrict__ q, int q_stride, const float* __restrict__ k_pool,
        const float* __restrict__ v_pool, PagedKV cache, int pages, const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, int n_heads, int group,
        float scale, int window, int sinks) {
    constexpr int DB = HD / 16, OWN = DB / 4;
    __shared__ f32x4 sums[4][DB][64];
    __shared__ float tops[4][16], dens[4][16];
    __shared__ unsigned ticket;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4, kvh = blockIdx.y;
    const int tiles = (group + 15) / 16, tok = blockIdx.x / tiles, first = 16 * (blockIdx.x - tok * tiles), rows = min(16, group);
    const bool real = first + i < group;
    const int head = kvh * group + min(first + i, group - 1), at = __builtin_amdgcn_readfirstlane(tok_pos[tok]), pos = real ? at : -1;
    const int seq = tok_seq ? tok_seq[tok] : tok, n_pages = min(at / kPageTokens + 1, pages), used = (n_pages + 3) / 4;
    if ((int)blockIdx.z >= used) return;
    auto unseen = [&](int page) { return window > 0 && page * kPageTokens >= sinks && page * kPageTokens + kPageTokens - 1 <= at - window; };
    const int page = 4 * blockIdx.z + wave;
    const bool seen = page < n_pages && !unseen(page);
    float m = -INFINITY, l = 0.f;
    f32x4 o[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (seen) {
        f32x8 qv[HD / 32];
#pragma unroll
        for (int d = 0; d < HD / 32; ++d)
            qv[d] = *reinterpret_cast<const f32x8*>(q + (size_t)tok * q_stride + (size_t)head * HD + 32 * d + 8 * g);
        const size_t base = paged_base(cache, seq, kvh, page * kPageTokens);
        attn_f32_page<HD>(k_pool + base, v_pool + base, qv, pos, at, page * kPageTokens, scale, window, sinks, m, l, o);
    }
    if (used == 1) {
#pragma unroll
        for (int d = 0; d < DB; ++d) sums[wave][d][lane] = o[d];
        if (g == 0) { tops[wave][i] = m; dens[wave][i] = l; }
        __syncthreads();
        f32x4 acc[OWN];
#pragma unroll
        for (int w = 0; w < OWN; ++w) acc[w] = f32x4{0.f, 0.f, 0.f, 0.f};
        float top = -INFINITY, den = 0.f;
        for (int j = 0; j < n_pages; ++j) {
            const float mj = tops[j][i], high = fmaxf(top, mj);
            const float keep = top == -INFINITY ? 0.f : expf(top - high), add = mj == -INFINITY ? 0.f : expf(mj - high);
#pragma unroll
            for (int w = 0; w < OWN; ++w) {
                const f32x4 v = sums[j][wave + 4 * w][lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[w][r] = fmaf(add == 0.f ? 0.f : v[r], add, (keep == 0.f ? 0.f : acc[w][r]) * keep);
            }
            den = fmaf(dens[j][i], add, den * keep);
            top = high;
        }
        const float inv = den > 0.f ? 1.0f / den : 0.f;
        if (!real) return;
#pragma unroll
        for (int w = 0; w < OWN; ++w) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[w][r] *= inv;
            *reinterpret_cast<f32x4*>(out + ((size_t)tok * n_heads + head) * HD + 16 * (wave + 4 * w) + 4 * g) = acc[w];
        }
        return;
    }
    const size_t mine = (size_t)blockIdx.x * gridDim.y + kvh;
    float* share0 = shares + mine * pages * attn_f32_share(rows, HD);
    if (seen && real) {
        float* share = share0 + (size_t)page * attn_f32_share(rows, HD);
#pragma unroll
        for (int d = 0; d < DB; ++d) {
            share_store(share + i * HD + 16 * d + 4 * g, o[d][0], o[d][1]);
            share_store(share + i * HD + 16 * d + 4 * g + 2, o[d][2], o[d][3]);
        }
        if (g == 0) share_store(share + rows * HD + 2 * i, m, l);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                     // this wave's share has arrived
    __syncthreads();                                                     // and every wave's
    if (threadIdx.x == 0) ticket = atomicInc(tickets + mine, (unsigned)used - 1);
    __syncthreads();
    if (ticket < (unsigned)used - 1) return;
    for (int idx = threadIdx.x; idx < min(rows, group - first) * (HD / 2); idx += 256) {
        const int row = idx / (HD / 2), c = 2 * (idx % (HD / 2));
        float2 v[kSharedPages], ml[kSharedPages];
#pragma unroll
        for (int j = 0; j < kSharedPages; ++j) {
            const float* share = share0 + (size_t)min(j, n_pages - 1) * attn_f32_share(rows, HD);
            v[j] = share_load(share + row * HD + c);
            ml[j] = share_load(share + rows * HD + 2 * row);
        }
        float top = -INFINITY, den = 0.f, x = 0.f, y = 0.f;
#pragma unroll
        for (int j = 0; j < kSharedPages; ++j) {
            if (j >= n_pages || unseen(j)) continue;
            const float mj = ml[j].x, high = fmaxf(top, mj);
            const float keep = top == -INFINITY ? 0.f : expf(top - high), add = mj == -INFINITY ? 0.f : expf(mj - high);
            x = fmaf(add == 0.f ? 0.f : v[j].x, add, (keep == 0.f ? 0.f : x) * keep);
            y = fmaf(add == 0.f ? 0.f : v[j].y, add, (keep == 0.f ? 0.f : y) * keep);
            den = fmaf(ml[j].y, add, den * keep);
            top = high;
        }
        const float inv = den > 0.f ? 1.0f / den : 0.f;
        *reinterpret_cast<float2*>(out + ((size_t)tok * n_heads + kvh * group + first + row) * HD + c) = make_float2(x * inv, y * inv);
    }
}

// n_tiles: tiles of 16 (token, head of the group) rows over all sequences, or more; pages: the most a sequence has (0: unknown); cu null:
// every sequence brings one token
LLOGOS_EXPORT int llogos_attention_f32(float* out, const float* q, int q_stride, const float* k_pool, const float* v_pool,
                                       const int* table, int table_stride, const int* cu, const int* tok_seq, const int* tok_pos,
                                       int batch, int n_tiles, int pages, int n_heads, int n_kv_heads, int head_dim, float scale, int window, int sinks,
                                       hipStream_t stream) {
    if (batch <= 0 || n_tiles <= 0 || n_kv_heads <= 0 || n_heads <= 0 || n_heads % n_kv_heads != 0 || window < 0 || sinks < 0) return LLOGOS_BAD_ARGUMENT;
    if ((head_dim != 64 && head_dim != 128) || (q_stride & 3) || (((uintptr_t)q | (uintptr_t)out) & 15)) return LLOGOS_UNSUPPORTED;
    const int group = n_heads / n_kv_heads;
    PagedKV cache{table, table_stride, n_kv_heads, head_dim};
    const dim3 grid(n_tiles, n_kv_heads);
    // Waves that share a tile's pages: many where there are few tiles (a single-token step: as many as LDS holds results of), few where
    // the tiles alone fill the GPU, and no more than there are pages: a wave without one still costs its block's start and its share
    // of LDS (64 sequences of 40 tokens, 32 heads of 128 by themselves: 62 us with four waves, 26 with one; 42 in the kernel for any shape).
    int waves = (long long)n_tiles * n_kv_heads >= 1024 ? 4 : (head_dim == 64 ? 16 : 8);
    while (waves > 1 && pages > 0 && waves / 2 >= pages) waves /= 2;
#define ATTN(HD, W) attn_f32_kernel<HD, W><<<grid, W * 64, 0, stream>>>(out, q, q_stride, k_pool, v_pool, cache, cu, batch, tok_seq, tok_pos, \
                                                                        n_heads, group, scale, window, sinks); break
#define BY_WAVES(HD) switch (waves) { case 1: ATTN(HD, 1); case 2: ATTN(HD, 2); case 4: ATTN(HD, 4); case 8: ATTN(HD, 8); default: ATTN(64, 16); }
    if (head_dim == 64) BY_WAVES(64)
    else BY_WAVES(128)
#undef BY_WAVES
#undef ATTN
    return LLOGOS_LAUNCH_CHECK();
}

LLOGOS_EXPORT long long llogos_attention_f32_pages_floats(int batch, int pages, int n_heads, int n_kv_heads, int head_dim) {
    if (batch <= 0 || pages <= 0 || n_kv_heads <= 0 || n_heads < n_kv_heads || n_heads % n_kv_heads || (head_dim != 64 && head_dim != 128)) return 0;
    const int group = n_heads / n_kv_heads;
    return (long long)batch * ((group + 15) / 16) * n_kv_heads * pages * attn_f32_share(group < 16 ? group : 16, head_dim);
}

// The same for one token a sequence with the pages side by side (attn_f32_pages_kernel), with the same bits; pages: those that a row of the table
// holds; shares: llogos_attention_f32_pages_floats floats; tickets: a counter for each sequence, tile of 16 heads of a group and kv head, zero before and
// after the call, with which up to kSharedPages pages take one kernel, or null.
LLOGOS_EXPORT int llogos_attention_f32_pages(float* out, float* shares, unsigned* tickets, const float* q, int q_stride, const float* k_pool, const float* v_pool,
                                             const int* table, int table_stride, int pages, const int* tok_seq, const int* tok_pos, int batch, int n_heads,
                                             int n_kv_heads, int head_dim, float scale, int window, int sinks, hipStream_t stream) {
    if (batch <= 0 || pages <= 0 || n_kv_heads <= 0 || n_kv_heads > 65535 || n_heads <= 0 || n_heads % n_kv_heads != 0 || window < 0 || sinks < 0) return LLOGOS_BAD_ARGUMENT;
    if ((head_dim != 64 && head_dim != 128) || (q_stride & 3) || (((uintptr_t)q | (uintptr_t)out | (uintptr_t)shares) & 15)) return LLOGOS_UNSUPPORTED;
    const int group = n_heads / n_kv_heads, n_tiles = batch * ((group + 15) / 16), rows = group < 16 ? group : 16;
    PagedKV cache{table, table_stride, n_kv_heads, head_dim};
    if (tickets && pages <= kSharedPages) {
#define SHARED(HD) attn_f32_shared_kernel<HD><<<dim3(n_tiles, n_kv_heads, (pages + 3) / 4), 256, 0, stream>>>(out, shares, tickets, q, q_stride, k_pool, v_pool, \
                                                                                        cache, pages, tok_seq, tok_pos, n_heads, group, scale, window, sinks)
        if (head_dim == 64) SHARED(64); else SHARED(128);
#undef SHARED
        return LLOGOS_LAUNCH_CHECK();
    }
    // about a wave for every matrix unit
    const long long across = (long long)n_tiles * n_kv_heads, want = (4LL * device_units() + across - 1) / across;
    const dim3 grid(n_tiles, n_kv_heads, (unsigned)(want < pages ? want : pages)), mgrid(n_tiles, n_kv_heads);
#define PAGES(HD) attn_f32_pages_kernel<HD><<<grid, 64, 0, stream>>>(shares, q, q_stride, k_pool, v_pool, cache, pages, tok_seq, tok_pos, group, scale, window, sinks); \
                  attn_f32_pages_merge<HD><<<mgrid, rows * (HD / 4), 0, stream>>>(out, shares, pages, tok_pos, n_heads, group, window, sinks)
    if (head_dim == 64) { PAGES(64); } else { PAGES(128); }
#undef PAGES
    return LLOGOS_LAUNCH_CHECK();
}
