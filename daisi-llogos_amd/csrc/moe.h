// What the products of experts share (moe.hip, moe_packed.hip).
#pragma once
#include "common.h"

// the two ways in which a gate and an up sum become one value: 2 silu(gate) * up; 3 with g = min(gate, limit) and
// u = up kept within -limit .. limit, g * sigmoid(1.702 g) * (u + 1)
__device__ __forceinline__ float moe_gated(float gate, float up, int act, float limit) {
    if (act == 3) {
        const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    return gate / (1.0f + expf(-gate)) * up;
}

__device__ __forceinline__ void moe_store4(float* p, float a, float b, float c, float d) {
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
}
__device__ __forceinline__ void moe_store4(bf16_t* p, float a, float b, float c, float d) {
    uint2 u;
    u.x = (uint32_t)f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16);
    u.y = (uint32_t)f32_to_bf16(c) | ((uint32_t)f32_to_bf16(d) << 16);
    *reinterpret_cast<uint2*>(p) = u;
}

__device__ __forceinline__ void moe_store2(float* p, float a, float b) { *reinterpret_cast<float2*>(p) = make_float2(a, b); }
__device__ __forceinline__ void moe_store2(bf16_t* p, float a, float b) {
    *reinterpret_cast<uint32_t*>(p) = (uint32_t)f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16);
}

// which tile of `rows` sorted rows is this block's: expert, first row, end of the expert's segment (expert -1: none).
// For one whole wave, whose lanes take the segments side by side: a thread that walks them waits for the cache once
// a segment, several microseconds before a block asks for its first weights.
__device__ __forceinline__ void moe_find_tile(const int* __restrict__ seg, int E, int rows, int tile, int& expert, int& first, int& end) {
    const int lane = threadIdx.x & (kWave - 1);
    expert = -1; first = 0; end = 0;
    for (int e0 = 0; e0 < E; e0 += kWave) {
        const int e = e0 + lane, lo = seg[min(e, E)], hi = seg[min(e + 1, E)];
        const int tiles = (hi - lo + rows - 1) / rows;
        int before = tiles;                                  // tiles of this segment and the ones in front of it
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) { const int v = __shfl_up(before, o, kWave); if (lane >= o) before += v; }
        const unsigned long long mine = __ballot(tile < before);
        if (mine) {
            const int at = __ffsll(mine) - 1;
            expert = e0 + at;
            end = __shfl(hi, at, kWave);
            first = __shfl(lo + (tile - (before - tiles)) * rows, at, kWave);
            return;
        }
        tile -= __shfl(before, kWave - 1, kWave);
    }
}
