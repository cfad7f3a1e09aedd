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
// tokens 14,731 -> 288; single tokens behind 515 and 190: 158 -> 17, behind 8,192: 2,625 -> 142.  Heads of 128: 1,496 -> 90,
// 19,143 -> 536, 180 -> 27, 2,721 -> 259.
// Behind only where a step's longest context has fewer than some 16 tokens, since a page is worked on whole: one token of heads
// of 64 by itself 4.9 -> 7.7, of 128 5.9 -> 11.3, a prompt of 16 11.2 -> 11.8 (the other kernel adds in another order, so
// serving those with it would cost the bits that a token has in common with itself in a longer step).
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8), aligned(16)));

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
