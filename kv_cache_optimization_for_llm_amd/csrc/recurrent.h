// What the kernels of the recurrent mixers share: loads and stores of either storage type, and the activations of
// decays, step sizes and gates.
#pragma once
#include "common.h"
#include <math.h>

__device__ inline float rec_ld(const void *p, int dtype, size_t i) {
    return dtype == KVA_BF16 ? bf16_bits_to_float(reinterpret_cast<const uint16_t *>(p)[i])
                             : reinterpret_cast<const float *>(p)[i];
}

__device__ inline void rec_st(void *p, int dtype, size_t i, float v) {
    if (dtype == KVA_BF16) reinterpret_cast<uint16_t *>(p)[i] = float_to_bf16_bits(v);
    else reinterpret_cast<float *>(p)[i] = v;
}

__device__ inline float rec_sigmoid(float z) { return 1.f / (1.f + expf(-z)); }
__device__ inline float rec_silu(float z) { return z / (1.f + expf(-z)); }
__device__ inline float rec_softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
__device__ inline float rec_act(float z, int act) { return act == 1 ? rec_silu(z) : z; }
