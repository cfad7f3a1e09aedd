// Token selection on the device, one block per row of logits.
//  - argmax: first maximum wins (reference: Daisi.Llogos/Inference/Sampler.cs:234-247).
//  - the sampling pipeline of Daisi.Llogos/Inference/Sampler.cs:26-85: penalties,
//    temperature, top-k, min-p, softmax over the candidates, typical-p, top-p and the
//    draw, which walks the candidates in descending order of their scaled logit (the
//    order in which the reference's top-k collection leaves them, :249-276) and takes
//    the first whose cumulative probability exceeds the uniform number (:334-345).
#include "common.h"

constexpr int kSampleThreads = 1024;

// f(i, row[i]) for every i < V, the block's threads together, in no particular order: eight
// 16-byte loads in flight per thread where the row allows them (one block reads a row of
// 10^5 values from the L2 in a few microseconds this way; one 4-byte load at a time, each
// waiting for the last, takes thirty).
template <typename F>
__device__ __forceinline__ void for_each_value(const float* __restrict__ row, int V, F f) {
    constexpr int U = 8;
    if ((V & 3) == 0 && ((uintptr_t)row & 15) == 0) {
        const float4* row4 = reinterpret_cast<const float4*>(row);
        const int n4 = V >> 2;
        for (int i0 = threadIdx.x; i0 < n4; i0 += U * blockDim.x) {
            float4 v[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int i = i0 + j * blockDim.x;
                v[j] = i < n4 ? row4[i] : float4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int i = i0 + j * blockDim.x;
                if (i < n4) { f(4 * i, v[j].x); f(4 * i + 1, v[j].y); f(4 * i + 2, v[j].z); f(4 * i + 3, v[j].w); }
            }
        }
    } else {
        for (int i0 = threadIdx.x; i0 < V; i0 += U * blockDim.x) {
            float v[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int i = i0 + j * blockDim.x;
                v[j] = i < V ? row[i] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int i = i0 + j * blockDim.x;
                if (i < V) f(i, v[j]);
            }
        }
    }
}

// ---------------------------------------------------------------- argmax
__global__ __launch_bounds__(kSampleThreads) void argmax_kernel(int* __restrict__ out,
                                                                const float* __restrict__ logits, int V) {
    __shared__ float s_val[kSampleThreads / kWave];
    __shared__ int s_idx[kSampleThreads / kWave];
    const float* row = logits + (size_t)blockIdx.x * V;
    float best = -INFINITY;
    int best_i = 0x7fffffff;
    if ((V & 3) == 0 && ((uintptr_t)row & 15) == 0) {
        // four values per load, several loads in flight; a thread visits its indices in
        // ascending order, so the strict comparison keeps the first maximum
        const float4* row4 = reinterpret_cast<const float4*>(row);
        const int n4 = V >> 2;
#pragma unroll 4
        for (int i = threadIdx.x; i < n4; i += blockDim.x) {
            const float4 v = row4[i];
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e[j] > best || best_i == 0x7fffffff) { best = e[j]; best_i = 4 * i + j; }
        }
    } else {
        for (int i = threadIdx.x; i < V; i += blockDim.x) {
            const float v = row[i];
            if (v > best || best_i == 0x7fffffff) { best = v; best_i = i; }
        }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o, kWave);
        const int oi = __shfl_xor(best_i, o, kWave);
        if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }
    }
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    if (lane == 0) { s_val[wave] = best; s_idx[wave] = best_i; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int wv = 1; wv < kSampleThreads / kWave; ++wv)
            if (s_val[wv] > best || (s_val[wv] == best && s_idx[wv] < best_i)) { best = s_val[wv]; best_i = s_idx[wv]; }
        out[blockIdx.x] = best_i;
    }
}

LLOGOS_EXPORT int llogos_argmax(int* out, const float* logits, int R, int V, hipStream_t stream) {
    if (R <= 0 || V <= 0) return LLOGOS_BAD_ARGUMENT;
    argmax_kernel<<<R, kSampleThreads, 0, stream>>>(out, logits, V);
    return LLOGOS_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- penalties and temperature
// work[r, :] = logits[r, :] with the repetition / frequency / presence penalties of the
// last `hist_len[r]` tokens applied (Sampler.cs:89-143: per occurrence l/p or l*p by sign,
// then - frequency * count - presence once per distinct token; tokens 10 and 13 are spared
// unless penalize_newline), the given ids set to -inf (PreventEOS, :49-53), then times
// 1 / temperature (:60-62).
constexpr int kMaxBanned = 64;           // ids that a call can ban (a model's stop tokens)
struct PenaltyParams {
    float repetition, frequency, presence, inv_temperature;
    int penalize_newline;
    int n_banned;
    int banned[kMaxBanned];
};

// The tokens of a window of n that lie in first .. first + count - 1 are made again from the logits, penalty first, then the scale.  A round's threads look at a position of the window each and list those
// that name such a token; a wave takes a listed position and reads the window 64 tokens at a time: a token's first occurrence
// does the work.  (One thread a position, reading the window token by token, made this 11 us of a slice's 16.)  put(q, place, value) takes
// the new value for first + place of a round's listed position q (place -1: an earlier position names the token), round() ends a round.
struct WindowLds {
    int n;
    int at[kSampleThreads];
};

// Adds to `times` how often a wave (lane) finds position i's token tok at positions BEGIN .. END - 1; where a position before i names it too, times is 0
// and LAST is done.  (As a loop each for LDS and memory: choosing for each position where to read, 64 windows of 8,000 tokens took 8 % longer.)
#define LLOGOS_COUNT_TOKEN(TOKEN, BEGIN, END, LAST) \
    for (int j0 = (BEGIN); j0 < (END); j0 += kWave) { \
        const uint64_t same = __ballot(j0 + lane < (END) && TOKEN(j0 + lane) == tok); \
        const uint64_t later = j0 >= i ? ~(uint64_t)0 : i - j0 >= kWave ? 0 : ~(uint64_t)0 << (i - j0); \
        if (same & ~later) { times = 0; LAST; break; } \
        times += (int)__popcll(same & later); \
    }

// token(i): the window's token at a position; times_of(i, tok): how often the window names position i's token, 0 where an earlier one does.
template <typename Token, typename Times, typename Put, typename Round>
__device__ __forceinline__ void apply_penalties(const float* __restrict__ row, int first, int count, int V, int n, const PenaltyParams& pp,
                                                WindowLds& lds, Token token, Times times_of, Put put, Round round) {
    const float inv_t = pp.inv_temperature;
    const bool scaled = inv_t != 1.0f;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, waves = blockDim.x / kWave;
    for (int i0 = 0; i0 < n; i0 += blockDim.x) {
        __syncthreads();
        if (threadIdx.x == 0) lds.n = 0;
        __syncthreads();
        if (i0 + (int)threadIdx.x < n) {
            const int i = i0 + threadIdx.x, tok = token(i);
            if (tok >= first && tok - first < count && tok < V && (pp.penalize_newline || (tok != 10 && tok != 13)))
                lds.at[atomicAdd(&lds.n, 1)] = i;
        }
        __syncthreads();
        for (int q = wave; q < lds.n; q += waves) {
            const int i = lds.at[q], tok = token(i), times = times_of(i, tok);
            if (lane != 0) continue;
            if (times == 0) { put(q, -1, 0.f); continue; }
            float l = row[tok];
            if (pp.repetition != 1.0f)
                for (int c = 0; c < times; ++c) l = l > 0.f ? l / pp.repetition : l * pp.repetition;
            if (pp.frequency != 0.f || pp.presence != 0.f) {
                l -= pp.frequency * (float)times;
                l -= pp.presence;
            }
            put(q, tok - first, scaled ? l * inv_t : l);
        }
        round();
    }
}

__device__ __forceinline__ bool has_penalties(const PenaltyParams& pp) {
    return pp.repetition != 1.0f || pp.frequency != 0.f || pp.presence != 0.f;
}

// a whole row by one block; h: the row's window of n tokens, or null
__device__ void prepare_row(float* w, const float* __restrict__ row, int V, const int* __restrict__ h, int n, const PenaltyParams& pp,
                            WindowLds& lds) {
    const float inv_t = pp.inv_temperature;
    const bool scaled = inv_t != 1.0f;
    for_each_value(row, V, [&](int i, float x) { w[i] = scaled ? x * inv_t : x; });
    __syncthreads();
    if (has_penalties(pp) && h) {
        const int lane = threadIdx.x & (kWave - 1);
        auto token = [&](int i) { return h[i]; };
        apply_penalties(row, 0, V, V, n, pp, lds, token, [&](int i, int tok) { int times = 0; LLOGOS_COUNT_TOKEN(token, 0, n, ) return times; },
                        [&](int, int place, float x) { if (place >= 0) w[place] = x; }, [] {});
        __syncthreads();
    }
    if (threadIdx.x < pp.n_banned) {
        const int tok = pp.banned[threadIdx.x];
        if (tok >= 0 && tok < V) w[tok] = -INFINITY;
    }
}

__global__ __launch_bounds__(kSampleThreads) void sample_prepare_kernel(
        float* __restrict__ work, const float* __restrict__ logits, int V,
        const int* __restrict__ hist, const int* __restrict__ hist_len, int hist_stride, PenaltyParams pp) {
    __shared__ WindowLds lds;
    const int r = blockIdx.x;
    prepare_row(work + (size_t)r * V, logits + (size_t)r * V, V, hist ? hist + (size_t)r * hist_stride : nullptr,
                hist ? hist_len[r] : 0, pp, lds);
}

LLOGOS_EXPORT int llogos_sample_prepare(float* work, const float* logits, int R, int V,
                                        const int* hist, const int* hist_len, int hist_stride,
                                        float repetition, float frequency, float presence, float inv_temperature,
                                        int penalize_newline, const int* banned, int n_banned, hipStream_t stream) {
    if (R <= 0 || V <= 0 || n_banned < 0 || n_banned > kMaxBanned) return LLOGOS_BAD_ARGUMENT;
    PenaltyParams pp{repetition, frequency, presence, inv_temperature, penalize_newline, n_banned, {}};
    for (int i = 0; i < n_banned; ++i) pp.banned[i] = banned[i];
    sample_prepare_kernel<<<R, kSampleThreads, 0, stream>>>(work, logits, V, hist, hist_len, hist_stride, pp);
    return LLOGOS_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- the candidate pipeline
// Order-preserving map of a float onto an unsigned integer (larger float, larger integer).
__device__ __forceinline__ uint32_t ordered_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if (u == 0x80000000u) u = 0;          // -0 equals +0: the lower id decides between them, as between other equals
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
// ascending sort of these puts the larger value first and, among equals, the lower id
__device__ __forceinline__ uint64_t desc_key(float v, int id) {
    return ((uint64_t)(~ordered_bits(v)) << 32) | (uint32_t)id;
}
__device__ __forceinline__ uint64_t asc_key(float v, int id) {
    return ((uint64_t)ordered_bits(v) << 32) | (uint32_t)id;
}
__device__ __forceinline__ int key_id(uint64_t k) { return (int)(uint32_t)k; }

// In-place ascending bitonic sort of n_pad (a power of two) keys by one block.
__device__ void bitonic_sort(uint64_t* d, int n_pad) {
    for (int k = 2; k <= n_pad; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < n_pad; i += blockDim.x) {
                const int p = i ^ j;
                if (p > i) {
                    const uint64_t a = d[i], b = d[p];
                    const bool up = (i & k) == 0;
                    if ((a > b) == up) { d[i] = b; d[p] = a; }
                }
            }
            __syncthreads();
        }
    }
}

// Sum of f(i) for i < n over the block; f is evaluated in chunks of consecutive i per thread.
template <typename F>
__device__ float block_sum_over(int n, float* red, F f) {
    const int chunk = (n + blockDim.x - 1) / blockDim.x;
    const int lo = min(n, (int)threadIdx.x * chunk), hi = min(n, lo + chunk);
    float s = 0.f;
#pragma unroll 8
    for (int i = lo; i < hi; ++i) s += f(i);
    return block_sum(s, red);
}

// Sum of f(row[i]) for i < V over the block, each thread adding the values it visits.
template <typename F>
__device__ float block_sum_values(const float* row, int V, float* red, F f) {
    float s = 0.f;
    for_each_value(row, V, [&](int, float x) { s += f(x); });
    return block_sum(s, red);
}

// First i < n (and i >= from) whose running sum of f exceeds `target` (or reaches it when
// `reach`); -1 when none does.  `scan` holds blockDim.x floats, `found` one int.
template <typename F>
__device__ int first_crossing(int n, int from, float target, bool reach, float* scan, int* found, F f) {
    const int chunk = (n + blockDim.x - 1) / blockDim.x;
    const int lo = min(n, (int)threadIdx.x * chunk), hi = min(n, lo + chunk);
    float s = 0.f;
#pragma unroll 8
    for (int i = lo; i < hi; ++i) s += f(i);
    __syncthreads();
    scan[threadIdx.x] = s;
    if (threadIdx.x == 0) *found = 0x7fffffff;
    __syncthreads();
    for (int o = 1; o < blockDim.x; o <<= 1) {          // inclusive scan over the threads' sums
        float add = threadIdx.x >= o ? scan[threadIdx.x - o] : 0.f;
        __syncthreads();
        scan[threadIdx.x] += add;
        __syncthreads();
    }
    float run = scan[threadIdx.x] - s;                   // sum before this thread's chunk
    for (int i = lo; i < hi; ++i) {
        run += f(i);
        const bool hit = reach ? run >= target : run > target;
        if (hit && i >= from) { atomicMin(found, i); break; }
    }
    __syncthreads();
    const int first = *found;
    return first == 0x7fffffff ? -1 : first;
}

struct SampleParams {
    int top_k;          // 0 = off
    float top_p;        // >= 1 = off
    float min_p;        // 0 = off
    float typical_p;    // >= 1 = off
    int min_keep;
};

// Steps 2 to 6 on a list whose first n_list keys are the row's tokens in descending order of
// their scaled logit (lower id first among equals); n of the row's V tokens are candidates
// after top-k.  With n_list < n the list is only the head of that order: the steps that look
// at every candidate (the count of min-p, the sum of the softmax) then walk the row itself,
// and -1 comes back when a cut or the draw lies beyond the head.  `src` holds the scaled
// logits; the candidates' probabilities go to `dst` (indexed by token; src itself or another
// row of V floats).  Returns the token drawn.
__device__ int pipeline_on_sorted(uint64_t* list, int n_list, int n, const float* src, float* dst, int V,
                                  const SampleParams& sp, float u, float* red, float* scan, int* found) {
    const int keep = max(sp.min_keep, 1);
    // 2. min-p on the scaled logits (Sampler.cs:157-174): the kept ones are a prefix
    const float top = src[key_id(list[0])];
    float thr = -INFINITY;
    if (sp.min_p > 0.f && sp.min_p < 1.f && n > keep) {
        thr = top + logf(sp.min_p);
        const float cnt = n <= n_list
            ? block_sum_over(n, red, [&](int i) { return src[key_id(list[i])] >= thr ? 1.f : 0.f; })
            : block_sum_values(src, V, red, [&](float x) { return x >= thr ? 1.f : 0.f; });
        n = max(keep, (int)cnt);
    }
    __syncthreads();

    // 3. softmax over the candidates (Sampler.cs:278-295)
    const float esum = n <= n_list
        ? block_sum_over(n, red, [&](int i) { return expf(src[key_id(list[i])] - top); })
        : block_sum_values(src, V, red, [&](float x) { return x >= thr ? expf(x - top) : 0.f; });
    const float inv = 1.0f / esum;
    __syncthreads();
    const int head = min(n, n_list);
    for (int i = threadIdx.x; i < head; i += blockDim.x) {
        const int t = key_id(list[i]);
        dst[t] = expf(src[t] - top) * inv;
    }
    __syncthreads();

    // 4. typical-p (Sampler.cs:182-230): by |(-log p) - entropy| ascending, keep until the
    //    cumulative probability reaches typical_p, renormalise
    bool resorted = false;
    if (sp.typical_p > 0.f && sp.typical_p < 1.f && n > keep) {
        if (n > n_list) return -1;
        const float ent = block_sum_over(n, red, [&](int i) {
            const float p = dst[key_id(list[i])];
            return p > 0.f ? -p * logf(p) : 0.f; });
        __syncthreads();
        int np2 = 1;
        while (np2 < n) np2 <<= 1;
        for (int i = threadIdx.x; i < np2; i += blockDim.x) {
            uint64_t k = ~(uint64_t)0;
            if (i < n) {
                const int t = key_id(list[i]);
                const float p = dst[t];
                const float lp = p > 0.f ? -logf(p) : 3.4028235e38f;
                k = asc_key(fabsf(lp - ent), t);
            }
            list[i] = k;
        }
        __syncthreads();
        bitonic_sort(list, np2);
        int cut = first_crossing(n, keep - 1, sp.typical_p, true, scan, found,
                                 [&](int i) { return dst[key_id(list[i])]; });
        if (cut >= 0) n = cut + 1;
        const float s = block_sum_over(n, red, [&](int i) { return dst[key_id(list[i])]; });
        __syncthreads();
        if (s > 0.f)
            for (int i = threadIdx.x; i < n; i += blockDim.x) dst[key_id(list[i])] *= 1.0f / s;
        __syncthreads();
        resorted = true;
    }

    // 5. top-p (Sampler.cs:297-332): by probability descending, cut after the first whose
    //    cumulative probability exceeds p, renormalise
    if (sp.top_p > 0.f && sp.top_p < 1.f) {
        if (resorted) {
            int np2 = 1;
            while (np2 < n) np2 <<= 1;
            for (int i = threadIdx.x; i < np2; i += blockDim.x) {
                uint64_t k = ~(uint64_t)0;
                if (i < n) { const int t = key_id(list[i]); k = desc_key(dst[t], t); }
                list[i] = k;
            }
            __syncthreads();
            bitonic_sort(list, np2);
        }
        int cut = first_crossing(min(n, n_list), keep - 1, sp.top_p, false, scan, found,
                                 [&](int i) { return dst[key_id(list[i])]; });
        if (cut >= 0) n = cut + 1;
        else if (n > n_list) return -1;
        const float s = block_sum_over(n, red, [&](int i) { return dst[key_id(list[i])]; });
        __syncthreads();
        if (s > 0.f)
            for (int i = threadIdx.x; i < n; i += blockDim.x) dst[key_id(list[i])] *= 1.0f / s;
        __syncthreads();
    }

    // 6. the draw (Sampler.cs:334-345): first candidate whose cumulative probability exceeds u
    int pick = first_crossing(min(n, n_list), 0, u, false, scan, found, [&](int i) { return dst[key_id(list[i])]; });
    if (pick < 0 && n > n_list) return -1;
    return key_id(list[pick >= 0 ? pick : 0]);
}

// The head of the descending order without sorting the row.  A histogram of the distance to
// the largest logit says which bins hold the first `want` tokens; those bins' tokens are
// gathered into LDS (any order) and sorted there by their full keys.  The distance is
// monotonic in the logit, so a bin boundary never separates equal values.  Bins are 1/64 wide
// down to 24 units below the largest and 1/4 wide from there to 151.75 units below; the last
// bin takes everything beyond, whose exp(logit - largest) is exactly 0 in float32, and NaN.
// Returns how many sorted keys `head` then holds (each at least as large as every token left
// out), or 0 when more than kHeadMax would be needed or the largest is not finite.
// *complete: the head holds every token outside the last bin, that is every token whose
// probability is not exactly 0.
constexpr int kHeadMax = 4096, kHeadBins = 2048, kFineBins = 1536;
constexpr float kFinePerUnit = 64.f, kCoarsePerUnit = 4.f;

__device__ __forceinline__ int head_bin(float top, float x) {
    const float d = top - x;
    if (d < (float)kFineBins / kFinePerUnit) return (int)(d * kFinePerUnit);
    const float e = (d - (float)kFineBins / kFinePerUnit) * kCoarsePerUnit;
    return e < (float)(kHeadBins - 1 - kFineBins) ? kFineBins + (int)e : kHeadBins - 1;   // NaN, -inf: the last bin
}

__device__ int sorted_head(uint64_t* head, const float* row, int V, int want, float* red, float* scan, int* bins,
                           int* counter, bool* complete) {
    float m = -INFINITY;
    for_each_value(row, V, [&](int, float x) { m = fmaxf(m, x); });
    const float top = block_max(m, red);
    if (!(top > -INFINITY && top < INFINITY)) return 0;
    for (int i = threadIdx.x; i < kHeadBins; i += blockDim.x) bins[i] = 0;
    if (threadIdx.x == 0) *counter = 0;
    __syncthreads();
    for_each_value(row, V, [&](int, float x) {
        const int b = head_bin(top, x);
        if (b < kHeadBins - 1) atomicAdd(&bins[b], 1);
    });
    __syncthreads();
    // last bin needed: the first whose running count reaches `want`, or the last one in use when
    // there are fewer tokens than that (thread t adds bins 2 t and 2 t + 1, a scan over the
    // threads gives the running counts; the last bin's counter is still 0 and takes the answer)
    static_assert(kHeadBins == 2 * kSampleThreads, "two bins a thread");
    int* run = reinterpret_cast<int*>(scan);
    const int a = bins[2 * threadIdx.x], b = bins[2 * threadIdx.x + 1];
    run[threadIdx.x] = a + b;
    __syncthreads();
    for (int o = 1; o < blockDim.x; o <<= 1) {
        const int add = threadIdx.x >= o ? run[threadIdx.x - o] : 0;
        __syncthreads();
        run[threadIdx.x] += add;
        __syncthreads();
    }
    const int incl = run[threadIdx.x], excl = incl - (a + b);
    const int outside_last = run[blockDim.x - 1];                        // >= 1: the largest itself
    want = min(want, outside_last);
    if (threadIdx.x == 0) bins[kHeadBins - 1] = -1;
    __syncthreads();
    if (excl < want && incl >= want) {
        const bool in_first = excl + a >= want;
        const int total = in_first ? excl + a : incl;
        bins[kHeadBins - 1] = total <= kHeadMax ? 2 * (int)threadIdx.x + (in_first ? 0 : 1) : -1;
    }
    __syncthreads();
    const int last = bins[kHeadBins - 1];
    if (last < 0) return 0;
    for_each_value(row, V, [&](int i, float x) {
        if (head_bin(top, x) <= last) head[atomicAdd(counter, 1)] = desc_key(x, i);
    });
    __syncthreads();
    const int n = *counter;
    *complete = n == outside_last;
    int np2 = 1;
    while (np2 < n) np2 <<= 1;
    for (int i = n + threadIdx.x; i < np2; i += blockDim.x) head[i] = ~(uint64_t)0;
    __syncthreads();
    bitonic_sort(head, np2);
    return n;
}

// One block per row.  `work` holds the penalised, temperature-scaled logits.
//  - try_head: the block tries with the sorted head of the row alone (in LDS; probabilities go
//    to `prob`, the logits stay as they are): all candidates when top-k leaves at most
//    kHeadMax / 2, else the first kHeadMax / 2 of the whole row.
//  - where that cannot decide (see pipeline_on_sorted and sorted_head), or without try_head:
//    with sort_here the block sorts the whole row into `list`, this row's scratch of n_pad
//    keys, and turns `work` into probabilities in place (slow: one compute unit sorts 10^5
//    keys in milliseconds); without sort_here it leaves out[row] = -1 for sample_sorted_kernel.
struct PipelineLds {
    float red[16];
    float scan[kSampleThreads];
    int found;
    int counter;
    int bins[kHeadBins];
    uint64_t head[kHeadMax];
};

// the token of one row, or -1 where it has to be sorted whole and sort_here is not set
__device__ int row_token(PipelineLds& s, float* work, float* prob, int V, uint64_t* list, int n_pad, float u,
                         const SampleParams& sp, int try_head, int sort_here) {
    const int n = (sp.top_k > 0 && sp.top_k < V) ? sp.top_k : V;
    if (try_head && (n <= kHeadMax / 2 || n == V)) {
        bool complete = false;
        const int n_head = sorted_head(s.head, work, V, min(n, kHeadMax / 2), s.red, s.scan, s.bins, &s.counter, &complete);
        if (n_head > 0) {
            // a complete head holds every candidate that can be drawn: the rest count for nothing
            const int token = pipeline_on_sorted(s.head, n_head, complete ? min(n, n_head) : n, work, prob, V, sp, u, s.red, s.scan, &s.found);
            if (token >= 0) return token;
        }
        __syncthreads();
    }
    if (!sort_here) return -1;
    // 1. all tokens in descending order of their scaled logit, lower id first among equals;
    //    the first k of them are the candidates (Sampler.cs:249-276)
    for (int i = threadIdx.x; i < n_pad; i += blockDim.x)
        list[i] = i < V ? desc_key(work[i], i) : ~(uint64_t)0;
    __syncthreads();
    bitonic_sort(list, n_pad);
    return pipeline_on_sorted(list, V, n, work, work, V, sp, u, s.red, s.scan, &s.found);
}

__global__ __launch_bounds__(kSampleThreads) void sample_pipeline_kernel(
        int* __restrict__ out, float* __restrict__ work_all, float* __restrict__ prob_all, int V,
        uint64_t* __restrict__ list_all, int n_pad, const float* __restrict__ uniforms, SampleParams sp,
        int try_head, int sort_here) {
    __shared__ PipelineLds s;
    const int r = blockIdx.x;
    const int token = row_token(s, work_all + (size_t)r * V, prob_all + (size_t)r * V, V, list_all + (size_t)r * n_pad, n_pad,
                                uniforms[r], sp, try_head, sort_here);
    if (threadIdx.x == 0) out[r] = token;
}

// ---- few candidates (top-k up to kFewCandidates): a row is read once, by many blocks.
//
// One block a row (the kernels above: a pass that prepares the row, then three that look for its head) left three quarters of
// the compute units idle at 64 rows and moved each row five times.  Here a block takes a slice of a row, prepares it in
// registers and keeps what may be among the row's first top-k (sample_slices_kernel).  A second kernel, one block a row, cuts the slices' lists (some tens of keys each) the same way against
// the row's largest, sorts what is left and draws.  Up to 64 candidates one wave does steps 2 to 6 without a barrier; its sums
// are the additions of the block's in the same order.  Whatever these lists cannot decide (an infinite value, thousands of
// values within a bin) is done again by the row's block in the general way.
// 64 rows of 128,256 logits, top-k 40, penalties: 76 us in the two kernels above, 20 here (13.0 + 6.8; one row 65 and 14).  Twice or four times as many,
// shorter slices at 64 rows took 4 and 11 us more.
constexpr int kFewCandidates = 256;      // largest top-k served
constexpr int kSliceThreads = 512;
constexpr int kSliceCap = 1024;          // keys a slice can hand on

// the first bin up to which `want` values lie, of counts of kHeadBins bins, by a block of THREADS; the last bin does not
// count.  *total: values up to it, *outside: all counted (0: none, then -1 comes back).  part: 16 ints of LDS, cut: 2.
template <int THREADS>
__device__ int cut_bin(const int* bins, int want, int* part, int* cut, int* total, int* outside) {
    constexpr int PER = kHeadBins / THREADS;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int c[PER], mine = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int b = threadIdx.x * PER + i;
        c[i] = b < kHeadBins - 1 ? bins[b] : 0;
        mine += c[i];
    }
    int incl = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int add = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += add;
    }
    if (lane == kWave - 1) part[wave] = incl;
    if (threadIdx.x == 0) { cut[0] = -1; cut[1] = 0; }
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < THREADS / kWave; ++w) {
        if (w < wave) before += part[w];
        all += part[w];
    }
    want = min(want, all);
    int run = before + incl - mine;
    if (want > 0 && run < want && run + mine >= want) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (run < want && run + c[i] >= want) { cut[0] = threadIdx.x * PER + i; cut[1] = run + c[i]; }
            run += c[i];
        }
    }
    __syncthreads();
    *total = cut[1];
    *outside = all;
    return cut[0];
}

// grid (slices, rows).  VPT values a thread.  counts, tops: [rows][slices]; keys: [rows][slices][kSliceCap].  count -1: more
// than kSliceCap keys, or a largest value that is not finite.  hist_at (or null): row r's window is hist[hist_at[r] .. hist_at[r + 1]).
//
// A block is a chain of short steps that wait, so all of a launch's blocks are to be on the units at once: 64 registers let 4 in.  A
// slice's list is cut without bins: a wave sorts its threads' own largest values and offers the (top_k / 8)-th (rounded up); the largest of
// the eight that top_k threads' values reach (the least one in any case) cuts the list, which a tenth to a half more than top_k values pass.
// 64 rows of 128,256 logits 13.0 us.  (19.3 with the slice's values patched in LDS, 97 registers, two rounds of blocks and the top_k-th of all
// threads' largest values found by counting them in bins: the additions to the few bins that they share, 1.9 us alone, took 5.3 with four
// blocks on a unit, and a bin for each value before it is listed 4.3.)
template <int VPT>
__global__ __launch_bounds__(kSliceThreads) __attribute__((amdgpu_waves_per_eu(8)))
void sample_slices_kernel(
        uint64_t* __restrict__ keys, int* __restrict__ counts, float* __restrict__ tops, const float* __restrict__ logits, int V,
        const int* __restrict__ hist, const int* __restrict__ hist_at, PenaltyParams pp, int top_k) {
    constexpr int kSlice = VPT * kSliceThreads, kWaves = kSliceThreads / kWave;
    __shared__ int lds[kHeadBins];                                // the window's tokens, then (where all values are counted) bins
    __shared__ int reached[kWaves][kWaves];
    __shared__ float wave_top[kWaves], wave_least[kWaves], patch[kSliceThreads];
    __shared__ int part[16], cut[2], counter, patch_at[kSliceThreads];
    __shared__ WindowLds window;
    const int s = blockIdx.x, r = blockIdx.y, at = r * gridDim.x + s;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const float* row = logits + (size_t)r * V;
    const int first = s * kSlice, count = min(kSlice, V - first);
    const float inv_t = pp.inv_temperature;
    const bool scaled = inv_t != 1.0f, penalties = has_penalties(pp) && hist_at != nullptr;
    const int* h = penalties ? hist + hist_at[r] : nullptr;
    const int n_hist = penalties ? hist_at[r + 1] - hist_at[r] : 0;
    const bool wide = (V & 3) == 0 && ((uintptr_t)logits & 15) == 0;   // then four neighbours a load, else threads side by side
    auto place = [&](int j) { return wide ? ((j >> 2) * kSliceThreads + threadIdx.x) * 4 + (j & 3) : j * kSliceThreads + (int)threadIdx.x; };
    float v[VPT];
    if (wide) {
#pragma unroll
        for (int j = 0; j < VPT; j += 4) {
            const int i = place(j);
            float4 t = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
            if (i < count) t = *reinterpret_cast<const float4*>(row + first + i);
            v[j] = t.x; v[j + 1] = t.y; v[j + 2] = t.z; v[j + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < VPT; ++j) v[j] = place(j) < count ? row[first + place(j)] : -INFINITY;
    }
    for (int i = threadIdx.x; i < min(n_hist, kHeadBins); i += kSliceThreads) lds[i] = h[i];
    if (threadIdx.x == 0) counter = 0;
#pragma unroll
    for (int j = 0; j < VPT; ++j) v[j] = scaled ? v[j] * inv_t : v[j];
    // the thread that holds the slice's value i, and in which of its places (above 16 bits); it takes a new value for it (`at` the same for all)
    auto holder = [&](unsigned i) {
        const unsigned n = wide ? i >> 2 : i;
        return n % kSliceThreads | (wide ? n / kSliceThreads * 4 + (i & 3) : n / kSliceThreads) << 16;
    };
    auto take = [&](unsigned at, float x) {
        if ((at & 0xffff) == threadIdx.x) v[at >> 16] = x;
    };
    if (penalties) {
        // A round's new values, 64 at a time: a wave passes over those that others hold.  (One after the other, each waited for in LDS by all
        // waves, they were 40 us of a draw's 144 where 512 tokens of a window lie in one slice; so it takes 111.)
        auto put = [&](int q, int i, float x) { patch_at[q] = i; patch[q] = x; };
        auto round = [&] {
            __syncthreads();
            for (int q0 = 0; q0 < window.n; q0 += kWave) {
                const int i = q0 + lane < window.n ? patch_at[q0 + lane] : -1;
                const int x = __float_as_int(patch[q0 + lane]);                // (of those behind the last nothing is used)
                const unsigned at = holder(i);
                for (uint64_t mine = __ballot(i >= 0 && (at & 0xffff) / kWave == wave); mine; mine &= mine - 1) {
                    const int l = __builtin_ctzll(mine);
                    take(__builtin_amdgcn_readlane(at, l), __int_as_float(__builtin_amdgcn_readlane(x, l)));
                }
            }
        };
        auto near = [&](int i) { return lds[i]; };
        auto far = [&](int i) { return h[i]; };
        const int n_near = min(n_hist, kHeadBins);
        apply_penalties(row, first, count, V, n_hist, pp, window, [&](int i) { return i < n_near ? near(i) : far(i); }, [&](int i, int tok) {
            int times = 0;
            bool more = n_near < n_hist;
            LLOGOS_COUNT_TOKEN(near, 0, n_near, more = false)
            if (more) { LLOGOS_COUNT_TOKEN(far, n_near, n_hist, ) }
            return times;
        }, put, round);
    }
    for (int i = 0; i < pp.n_banned; ++i) {
        const int tok = pp.banned[i] - first;
        if (tok >= 0 && tok < count) take(holder(tok), -INFINITY);
    }
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < VPT; ++j) m = fmaxf(m, v[j]);              // (places past the slice hold -inf)
    // the wave's 64 largest values of a thread in falling order (bitonic): lane l has the l-th
    float sorted = m;
#pragma unroll
    for (int size = 2; size <= kWave; size <<= 1)
#pragma unroll
        for (int o = size >> 1; o > 0; o >>= 1) {
            const float other = __shfl_xor(sorted, o, kWave);
            const bool larger = ((lane & o) == 0) == ((lane & size) == 0);
            sorted = larger ? fmaxf(sorted, other) : fminf(sorted, other);
        }
    // (waves whose threads all have values; the others' values are listed like any)
    const int full = min(kWaves, (wide ? count >> 2 : count) / kWave), share = full > 0 ? (top_k + full - 1) / full : kWave + 1;
    if (lane == 0) wave_top[wave] = sorted;
    if (lane == min(share, kWave) - 1) wave_least[wave] = wave < full && share <= kWave ? sorted : -INFINITY;
    __syncthreads();
    float top = wave_top[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) top = fmaxf(top, wave_top[w]);
    // the largest of the waves' that top_k threads' largest values reach: their least one in any case
    {
        int reach = 0;                                            // lane w: how many of this wave's reach wave w's
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int n = (int)__popcll(__ballot(m >= wave_least[w]));
            reach = lane == w ? n : reach;
        }
        if (lane < kWaves) reached[wave][lane] = reach;
    }
    __syncthreads();
    float least = -INFINITY;
    if (lane < kWaves) {
        int n = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) n += reached[w][lane];
        if (n >= top_k) least = wave_least[lane];
    }
    least = wave_max(least);
    if (!(top > -INFINITY && top < INFINITY)) {
        if (threadIdx.x == 0) { counts[at] = top < INFINITY ? 0 : -1; tops[at] = top; }
        return;
    }
    auto list = [&](int j) {
        const int slot = atomicAdd(&counter, 1);
        if (slot < kSliceCap) keys[(size_t)at * kSliceCap + slot] = desc_key(v[j], first + place(j));
    };
    if (least > -INFINITY) {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
            if (v[j] >= least) list(j);
        __syncthreads();
        if (counter <= kSliceCap) {
            if (threadIdx.x == 0) { counts[at] = counter; tops[at] = top; }
            return;
        }
    }
    // Where a wave has fewer threads with a value than that, or the list would overflow: all values by the distance to the largest.
    __syncthreads();
    for (int i = threadIdx.x; i < kHeadBins; i += kSliceThreads) lds[i] = 0;
    if (threadIdx.x == 0) counter = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int b = head_bin(top, v[j]);
        if (b < kHeadBins - 1) atomicAdd(&lds[b], 1);
    }
    __syncthreads();
    int total, outside;
    const int last = cut_bin<kSliceThreads>(lds, top_k, part, cut, &total, &outside);
    const bool fits = total <= kSliceCap;
    if (fits) {
#pragma unroll
        for (int j = 0; j < VPT; ++j)
            if (head_bin(top, v[j]) <= last) list(j);
        __syncthreads();
    }
    if (threadIdx.x == 0) { counts[at] = fits ? counter : -1; tops[at] = top; }
}

__device__ __forceinline__ float key_value(uint64_t k) {            // of a desc_key (-0 comes back as 0)
    const uint32_t o = ~(uint32_t)(k >> 32);
    return __uint_as_float(o & 0x80000000u ? o & 0x7fffffffu : ~o);
}

// Steps 2, 3, 5 and 6 of pipeline_on_sorted for n <= 64 PER candidates, sorted in head, by one wave: value j of lane l is the
// (64 j + l)-th.  The same sums in the same order: a wave's sums one after the other as block_sum adds them, and the scan over
// the values step by step.
template <int PER>
__device__ int pipeline_on_wave(const uint64_t* head, int n, const SampleParams& sp, float u) {
    const int lane = threadIdx.x & (kWave - 1);
    const int keep = max(sp.min_keep, 1);
    const float top = key_value(head[0]);
    float x[PER], p[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) x[j] = key_value(head[min(j * kWave + lane, n - 1)]);
    auto sum_of = [&](const float (&f)[PER]) {
        float t = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j) t += wave_sum(j * kWave + lane < n ? f[j] : 0.f);
        return t;
    };
    if (sp.min_p > 0.f && sp.min_p < 1.f && n > keep) {
        const float thr = top + logf(sp.min_p);
        int kept = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) kept += (int)__popcll(__ballot(j * kWave + lane < n && x[j] >= thr));
        n = max(keep, kept);
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) p[j] = expf(x[j] - top);
    const float inv = 1.0f / sum_of(p);
#pragma unroll
    for (int j = 0; j < PER; ++j) p[j] = expf(x[j] - top) * inv;
    auto crossing = [&](int from, float target) {                    // first i >= from whose running sum exceeds target
        float incl[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) incl[j] = j * kWave + lane < n ? p[j] : 0.f;
#pragma unroll
        for (int o = 1; o < PER * kWave; o <<= 1) {
            float add[PER];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                if (o >= kWave) add[j] = j >= o / kWave ? incl[j - o / kWave] : 0.f;
                else {
                    const float same = __shfl(incl[j], lane - o, kWave), before = j > 0 ? __shfl(incl[j - 1], lane - o + kWave, kWave) : 0.f;
                    add[j] = lane >= o ? same : before;
                }
            }
#pragma unroll
            for (int j = 0; j < PER; ++j) incl[j] += add[j];
        }
        int first = -1;
#pragma unroll
        for (int j = PER - 1; j >= 0; --j) {
            const int i = j * kWave + lane;
            const float own = i < n ? p[j] : 0.f;
            float run = incl[j] - own;
            run += own;
            const uint64_t hits = __ballot(i < n && i >= from && run > target);
            if (hits) first = j * kWave + __ffsll((unsigned long long)hits) - 1;
        }
        return first;
    };
    if (sp.top_p > 0.f && sp.top_p < 1.f) {
        const int cut = crossing(keep - 1, sp.top_p);
        if (cut >= 0) n = cut + 1;
        const float sum = sum_of(p);
        if (sum > 0.f) {
#pragma unroll
            for (int j = 0; j < PER; ++j) p[j] *= 1.0f / sum;
        }
    }
    const int pick = crossing(0, u);
    return key_id(head[pick >= 0 ? pick : 0]);
}

// One block a row.  work, prob [rows][V] and list [rows][n_pad]: scratch that is written only where a row has to be done in the
// general way, or for typical-p.
__global__ __launch_bounds__(kSampleThreads) void sample_few_kernel(
        int* __restrict__ out, const uint64_t* __restrict__ keys, const int* __restrict__ counts, const float* __restrict__ tops, int slices,
        const float* __restrict__ logits, int V, const int* __restrict__ hist, const int* __restrict__ hist_at, PenaltyParams pp,
        float* __restrict__ work_all, float* __restrict__ prob_all, uint64_t* __restrict__ list_all, int n_pad,
        const float* __restrict__ uniforms, SampleParams sp) {
    __shared__ PipelineLds s;
    __shared__ WindowLds window;
    __shared__ int part[16], cut[2], slice_at[kWave + 1];
    const int r = blockIdx.x, lane = threadIdx.x & (kWave - 1);
    float* work = work_all + (size_t)r * V;
    float* prob = prob_all + (size_t)r * V;
    const float u = uniforms[r];
    for (int i = threadIdx.x; i < kHeadBins; i += kSampleThreads) s.bins[i] = 0;
    if (threadIdx.x == 0) s.counter = 0;
    // where each slice's keys go among the row's (slices <= kWave): every wave for itself, the first one for all
    const int mine = lane < slices ? counts[(size_t)r * slices + lane] : 0;
    const float top = wave_max(lane < slices ? tops[(size_t)r * slices + lane] : -INFINITY);
    const bool lost = __any(mine < 0) || !(top > -INFINITY && top < INFINITY);
    int incl = max(mine, 0);
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int add = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += add;
    }
    const int n_keys = __shfl(incl, kWave - 1, kWave);
    if (threadIdx.x < kWave) slice_at[lane + 1] = incl;
    if (threadIdx.x == 0) slice_at[0] = 0;
    __syncthreads();
    constexpr int PER = kWave * kFewCandidates / kSampleThreads;     // as many keys as slices of kFewCandidates each bring, for one
    if (!lost && n_keys <= PER * kSampleThreads) {
        uint64_t key[PER];
        int bin[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = j * kSampleThreads + threadIdx.x;
            bin[j] = kHeadBins;
            if (i < n_keys) {
                int at = 0;                                          // the slice whose run holds i: slice_at[at] <= i < slice_at[at + 1]
#pragma unroll
                for (int step = kWave / 2; step > 0; step >>= 1) if (slice_at[at + step] <= i) at += step;
                key[j] = keys[((size_t)r * slices + at) * kSliceCap + (i - slice_at[at])];
            }
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            if (j * kSampleThreads + (int)threadIdx.x >= n_keys) break;
            bin[j] = head_bin(top, key_value(key[j]));
            if (bin[j] < kHeadBins - 1) atomicAdd(&s.bins[bin[j]], 1);
        }
        __syncthreads();
        int total, outside;
        const int last = cut_bin<kSampleThreads>(s.bins, sp.top_k, part, cut, &total, &outside);
        if (total <= kHeadMax) {
        const int n = min(sp.top_k, total);                          // fewer only where fewer have a probability that is not 0
        // the keys up to that bin, in any order, then each to its rank (all keys differ)
        uint64_t* some = total <= kHeadMax / 2 ? s.head + kHeadMax / 2 : s.head;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (bin[j] <= last) some[atomicAdd(&s.counter, 1)] = key[j];
        __syncthreads();
        if (total <= kSampleThreads) {
            if (threadIdx.x < total) {
                const uint64_t k = some[threadIdx.x];
                int rank = 0;
                for (int i = 0; i < total; ++i) rank += some[i] < k;
                s.head[rank] = k;
            }
            __syncthreads();
        } else {
            if (some != s.head) {
                for (int i = threadIdx.x; i < total; i += kSampleThreads) s.head[i] = some[i];
                __syncthreads();
            }
            int np2 = 1;
            while (np2 < total) np2 <<= 1;
            for (int i = total + threadIdx.x; i < np2; i += kSampleThreads) s.head[i] = ~(uint64_t)0;
            __syncthreads();
            bitonic_sort(s.head, np2);
        }
        int token;
        if (!(sp.typical_p > 0.f && sp.typical_p < 1.f)) {
            if (threadIdx.x >= kWave) return;
            token = n <= kWave ? pipeline_on_wave<1>(s.head, n, sp, u) : n <= 2 * kWave ? pipeline_on_wave<2>(s.head, n, sp, u)
                                                                                      : pipeline_on_wave<kFewCandidates / kWave>(s.head, n, sp, u);
        } else {
            for (int i = threadIdx.x; i < n; i += kSampleThreads) work[key_id(s.head[i])] = key_value(s.head[i]);
            __syncthreads();
            token = pipeline_on_sorted(s.head, total, n, work, prob, V, sp, u, s.red, s.scan, &s.found);
        }
        if (threadIdx.x == 0) out[r] = token;
        return;
        }
    }
    prepare_row(work, logits + (size_t)r * V, V, hist_at ? hist + hist_at[r] : nullptr, hist_at ? hist_at[r + 1] - hist_at[r] : 0, pp, window);
    __syncthreads();
    const int token = row_token(s, work, prob, V, list_all + (size_t)r * n_pad, n_pad, u, sp, 1, 1);
    if (threadIdx.x == 0) out[r] = token;
}

// ---- whole rows sorted by many blocks: the bitonic network over n_pad keys, cut into chunks
// of kSortChunk keys that a block sorts or merges in LDS, and passes over global memory for the
// exchanges between chunks.  grid (chunks or blocks of pairs, rows); rows that already have
// their token (out[row] >= 0) are left alone.
constexpr int kSortChunk = 8192;

// the t-th pair (i, i + j) of an exchange at distance j: t with a zero bit put in at j's place
__device__ __forceinline__ int pair_low(int t, int j) { return ((t & ~(j - 1)) << 1) | (t & (j - 1)); }   // j: a power of two

__device__ __forceinline__ void exchange(uint64_t* d, int i, int p, bool up) {
    const uint64_t a = d[i], b = d[p];
    if ((a > b) == up) { d[i] = b; d[p] = a; }
}

// stage 0: makes the chunk's keys from the row and sorts it (network stages 2 .. chunk);
// stage k > chunk: the exchanges at distances chunk / 2 .. 1 of network stage k.
__global__ __launch_bounds__(kSampleThreads) void sort_chunk_kernel(
        uint64_t* __restrict__ list_all, const float* __restrict__ work_all, const int* __restrict__ out,
        int V, int n_pad, int stage) {
    __shared__ uint64_t d[kSortChunk];
    const int r = blockIdx.y;
    if (out[r] >= 0) return;
    const int m = min(kSortChunk, n_pad), base = blockIdx.x * m;
    uint64_t* list = list_all + (size_t)r * n_pad + base;
    if (stage == 0) {
        const float* work = work_all + (size_t)r * V;
        for (int i = threadIdx.x; i < m; i += blockDim.x)
            d[i] = base + i < V ? desc_key(work[base + i], base + i) : ~(uint64_t)0;
    } else {
        for (int i = threadIdx.x; i < m; i += blockDim.x) d[i] = list[i];
    }
    __syncthreads();
    for (int k = stage == 0 ? 2 : stage; k <= (stage == 0 ? m : stage); k <<= 1)
        for (int j = min(k, m) >> 1; j > 0; j >>= 1) {
            for (int t = threadIdx.x; t < m / 2; t += blockDim.x) {
                const int i = pair_low(t, j);
                exchange(d, i, i + j, ((base + i) & k) == 0);
            }
            __syncthreads();
        }
    for (int i = threadIdx.x; i < m; i += blockDim.x) list[i] = d[i];
}

// the exchanges at distance j >= chunk of network stage k
__global__ __launch_bounds__(kSampleThreads) void sort_exchange_kernel(
        uint64_t* __restrict__ list_all, const int* __restrict__ out, int n_pad, int k, int j) {
    const int r = blockIdx.y;
    if (out[r] >= 0) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_pad / 2) return;
    const int i = pair_low(t, j);
    exchange(list_all + (size_t)r * n_pad, i, i + j, (i & k) == 0);
}

// steps 2 to 6 for the rows sorted so; `work` becomes probabilities in place
__global__ __launch_bounds__(kSampleThreads) void sample_sorted_kernel(
        int* __restrict__ out, float* __restrict__ work_all, int V, uint64_t* __restrict__ list_all, int n_pad,
        const float* __restrict__ uniforms, SampleParams sp) {
    __shared__ float red[16];
    __shared__ float scan[kSampleThreads];
    __shared__ int found;
    const int r = blockIdx.x;
    if (out[r] >= 0) return;
    float* work = work_all + (size_t)r * V;
    const int n = (sp.top_k > 0 && sp.top_k < V) ? sp.top_k : V;
    const int token = pipeline_on_sorted(list_all + (size_t)r * n_pad, V, n, work, work, V, sp, uniforms[r], red, scan,
                                         &found);
    if (threadIdx.x == 0) out[r] = token;
}

// mode: 0 = every row sorted whole by its own block (the plain form); 1 = the head of the order
// first, rows it cannot decide sorted whole by many blocks; 2 = every row sorted by many blocks.
// In mode 1 the kernels of the many-block sort are launched only where an ordinary row can need
// them (no top-k, or one beyond the head's size); a row whose head is undecided although top-k
// is small (thousands of tokens within 1/64 of the k-th) is sorted by its own block.
LLOGOS_EXPORT int llogos_sample_pipeline(int* out, float* work, float* prob, int R, int V, void* list, int n_pad,
                                         const float* uniforms, int top_k, float top_p, float min_p,
                                         float typical_p, int min_keep, int mode, hipStream_t stream) {
    if (R <= 0 || V <= 0 || n_pad < V || (n_pad & (n_pad - 1)) || mode < 0 || mode > 2 || (mode == 1 && prob == nullptr))
        return LLOGOS_BAD_ARGUMENT;
    SampleParams sp{top_k, top_p, min_p, typical_p, min_keep};
    const int n = (top_k > 0 && top_k < V) ? top_k : V;
    const bool head_fits = n <= kHeadMax / 2 || n == V;
    const bool many_blocks = mode == 2 || (mode == 1 && (n == V || !head_fits));
    sample_pipeline_kernel<<<R, kSampleThreads, 0, stream>>>(out, work, prob, V, (uint64_t*)list, n_pad, uniforms, sp,
                                                             mode == 1, !many_blocks);
    if (many_blocks) {
        uint64_t* keys = (uint64_t*)list;
        const int m = n_pad < kSortChunk ? n_pad : kSortChunk;
        const dim3 chunks(n_pad / m, R), pairs((n_pad / 2 + kSampleThreads - 1) / kSampleThreads, R);
        sort_chunk_kernel<<<chunks, kSampleThreads, 0, stream>>>(keys, work, out, V, n_pad, 0);
        for (int k = 2 * m; k <= n_pad; k <<= 1) {
            for (int j = k >> 1; j >= m; j >>= 1)
                sort_exchange_kernel<<<pairs, kSampleThreads, 0, stream>>>(keys, out, n_pad, k, j);
            sort_chunk_kernel<<<chunks, kSampleThreads, 0, stream>>>(keys, work, out, V, n_pad, k);
        }
        sample_sorted_kernel<<<R, kSampleThreads, 0, stream>>>(out, work, V, keys, n_pad, uniforms, sp);
    }
    return LLOGOS_LAUNCH_CHECK();
}

// values a slice: small ones where there are few rows, at most kWave slices a row and no more keys of a row than sample_few_kernel takes
static int slice_values(int R, int V, int top_k) {
    auto slices = [&](int vpt) { return (V + vpt * kSliceThreads - 1) / (vpt * kSliceThreads); };
    int vpt = 4;
    while (vpt < 16 && ((long long)R * slices(vpt) > 1024 || slices(vpt) > kWave || slices(vpt) * top_k > kWave * kFewCandidates / 2)) vpt *= 2;
    return vpt * kSliceThreads;
}

// slices a row, 0: not served: among others more rows than a grid is high
static int few_slices(int R, int V, int top_k) {
    if (R <= 0 || R > 65535 || V <= 0 || top_k <= 0 || top_k > kFewCandidates || top_k >= V) return 0;
    const int values = slice_values(R, V, top_k), slices = (V + values - 1) / values;
    return slices <= kWave ? slices : 0;
}

// Preparation and pipeline of rows of which at most top_k <= kFewCandidates tokens can be drawn: the tokens that llogos_sample_prepare
// and llogos_sample_pipeline give.  keys [R][slices][cap] uint64, counts [R][slices], tops [R][slices]: scratch; work, prob [R][V] and
// list [R][n_pad]: scratch of the rows that need the general way.  hist_at (or null): offsets [R + 1] of the rows' windows in hist.
static int sample_few(int* out, const float* logits, int R, int V, const int* hist, const int* hist_at, float repetition, float frequency,
                      float presence, float inv_temperature, int penalize_newline, const int* banned, int n_banned, void* keys, int* counts,
                      float* tops, float* work, float* prob, void* list, int n_pad, const float* uniforms, int top_k, float top_p,
                      float min_p, float typical_p, int min_keep, hipStream_t stream) {
    const int slices = few_slices(R, V, top_k);
    if (slices == 0 || n_banned < 0 || n_banned > kMaxBanned || n_pad < V || (n_pad & (n_pad - 1))) return LLOGOS_BAD_ARGUMENT;
    PenaltyParams pp{repetition, frequency, presence, inv_temperature, penalize_newline, n_banned, {}};
    for (int i = 0; i < n_banned; ++i) pp.banned[i] = banned[i];
    const SampleParams sp{top_k, top_p, min_p, typical_p, min_keep};
    const dim3 grid(slices, R);
#define GO(VPT) sample_slices_kernel<VPT><<<grid, kSliceThreads, 0, stream>>>((uint64_t*)keys, counts, tops, logits, V, hist, hist_at, pp, top_k)
    const int vpt = slice_values(R, V, top_k) / kSliceThreads;
    if (vpt == 4) GO(4); else if (vpt == 8) GO(8); else GO(16);
#undef GO
    sample_few_kernel<<<R, kSampleThreads, 0, stream>>>(out, (const uint64_t*)keys, counts, tops, slices, logits, V, hist, hist_at, pp,
                                                        work, prob, (uint64_t*)list, n_pad, uniforms, sp);
    return LLOGOS_LAUNCH_CHECK();
}

// A sampler's settings, as its calls share them.
struct SampleSettings {
    float repetition, frequency, presence, inv_temperature, top_p, min_p, typical_p;
    int penalize_newline, top_k, min_keep, n_banned;
    int banned[kMaxBanned];
};

// 8-byte words of scratch memory for llogos_sample_few_staged beside the staged numbers; 0 where it does not serve
LLOGOS_EXPORT long long llogos_sample_few_words(int R, int V, int top_k) {
    const long long slices = few_slices(R, V, top_k);
    if (slices == 0) return 0;
    long long n_pad = 1;
    while (n_pad < V) n_pad *= 2;
    return R * slices * kSliceCap + R * n_pad + (long long)R * V + R * slices;
}

LLOGOS_EXPORT int llogos_copy_words(void* dst, const void* src, long long n, hipStream_t stream);     // (elementwise.hip)

// sample_few from what the host has packed into pinned memory: R uniform numbers (float32) and, with `windows`, the R + 1 places of the
// rows' windows and the windows, `staged` 32-bit numbers in all.  They are copied behind the scratch (16-byte aligned: llogos_sample_few_words words, then
// `staged` numbers), `copied` (an event or null) is recorded behind the copy, and the two kernels follow: one call for what a step of
// the sampler queues.
LLOGOS_EXPORT int llogos_sample_few_staged(int* out, const float* logits, int R, int V, const void* host, long long staged, int windows,
                                           const void* settings, void* scratch, void* copied, hipStream_t stream) {
    const SampleSettings* s = (const SampleSettings*)settings;
    if (s == nullptr || host == nullptr || scratch == nullptr || staged < R + (windows ? R + 1 : 0)) return LLOGOS_BAD_ARGUMENT;
    const long long slices = few_slices(R, V, s->top_k), words = llogos_sample_few_words(R, V, s->top_k);
    if (words == 0) return LLOGOS_BAD_ARGUMENT;
    long long n_pad = 1;
    while (n_pad < V) n_pad *= 2;
    uint64_t* keys = (uint64_t*)scratch;
    uint64_t* list = keys + R * slices * kSliceCap;
    float* work = (float*)(list + R * n_pad);
    float* prob = work + (size_t)R * V;
    int* counts = (int*)(prob + (size_t)R * V);
    float* tops = (float*)(counts + R * slices);
    int* numbers = (int*)(keys + words);
    const int code = llogos_copy_words(numbers, host, staged, stream);
    if (code != 0) return code;
    if (copied != nullptr) {
        const hipError_t e = hipEventRecord((hipEvent_t)copied, stream);
        if (e != hipSuccess) return (int)e;
    }
    return sample_few(out, logits, R, V, windows ? numbers + 2 * R + 1 : nullptr, windows ? numbers + R : nullptr, s->repetition, s->frequency,
                             s->presence, s->inv_temperature, s->penalize_newline, s->banned, s->n_banned, keys, counts, tops, work, prob, list,
                             (int)n_pad, (const float*)numbers, s->top_k, s->top_p, s->min_p, s->typical_p, s->min_keep, stream);
}
