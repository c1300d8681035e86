// Elementwise activations by number, alone or over pairs of neighbouring columns (a gate and an up value).
#pragma once
#include "common.h"

#define ACT_NONE 0
#define ACT_RELU2 1
#define ACT_SILU 2
#define ACT_GELU_TANH 3
#define ACT_GELU 4        // the exact form, with the error function
#define ACT_PAIRS 16      // added to one of the above: the product's columns 2i and 2i + 1 are a gate and an up value, the output act(gate) * up

__device__ __forceinline__ float activate(float v, int act) {
    if (act == ACT_RELU2) { v = fmaxf(v, 0.f); return v * v; }
    if (act == ACT_SILU) return v / (1.f + expf(-v));
    if (act == ACT_GELU_TANH) return gelu_tanh(v);
    if (act == ACT_GELU) return 0.5f * v * (1.f + erff(v * 0.7071067811865476f));
    return v;
}

__host__ __device__ __forceinline__ bool known_activation(int act) { return (act & ~ACT_PAIRS) >= ACT_NONE && (act & ~ACT_PAIRS) <= ACT_GELU; }
