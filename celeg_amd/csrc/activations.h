// The activations that follow a product, in 32-bit: as kernels of their own and inside a product's epilogue.
#pragma once
#include "common.h"

enum CelegActivation { CELEG_ACT_GELU_TANH = 0, CELEG_ACT_RELU2 = 1, CELEG_ACT_NONE = 2, CELEG_ACT_BENT = 3 };

__device__ __forceinline__ float lg_gelu_tanh(float z) {
    // 0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3)))
    const float inner = 0.7978845608028654f * (z + 0.044715f * z * z * z);
    return 0.5f * z * (1.0f + tanhf(inner));
}
__device__ __forceinline__ float lg_relu2(float z) {
    const float r = fmaxf(z, 0.f);
    return r * r;
}

// z > 0: right z^2 + z / 2;  z <= 0: left (exp(z) - 1 - z) + z / 2 (both pieces and their slopes meet at 0)
__device__ __forceinline__ float lg_bent(float z, float right, float left) {
    return (z > 0.f ? right * z * z : left * (expm1f(z) - z)) + 0.5f * z;
}

__device__ __forceinline__ float activated(float z, int act, float p0, float p1) {
    return act == CELEG_ACT_GELU_TANH ? lg_gelu_tanh(z) : act == CELEG_ACT_RELU2 ? lg_relu2(z) : act == CELEG_ACT_BENT ? lg_bent(z, p0, p1) : z;
}
