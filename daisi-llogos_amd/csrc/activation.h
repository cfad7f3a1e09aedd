// Activations of a product, for the kernel that applies them (sequence_state.hip) and the products that do so themselves (gemm_tiles.h).  kinds:
//   0 tanh;  1 silu;  2 gelu (tanh form);
//   3 the piecewise xIELU with a = softplus(p), b = 1/2 + softplus(q):
//       z > 0: a z^2 + z / 2;   z <= 0: b (exp(z) - 1 - z) + z / 2
//   4 the square of relu: max(z, 0)^2;  5 the sum as it is
#pragma once
#include "common.h"

enum { ACT_TANH = 0, ACT_SILU = 1, ACT_GELU_TANH = 2, ACT_XIELU = 3, ACT_RELU2 = 4, ACT_NONE = 5 };

__device__ __forceinline__ float activate(float z, int kind, float a, float b) {
    switch (kind) {
        case ACT_TANH: return tanhf(z);
        case ACT_SILU: return z / (1.0f + expf(-z));
        case ACT_GELU_TANH: return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
        case ACT_RELU2: { const float r = fmaxf(z, 0.f); return r * r; }
        case ACT_NONE: return z;
        default: return z > 0.f ? fmaf(a * z, z, 0.5f * z) : fmaf(b, expm1f(z) - z, 0.5f * z);
    }
}
