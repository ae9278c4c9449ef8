// What the kernels of the recurrent mixers share: loads and stores of either storage type, and the activations of
// decays, step sizes and gates.
#pragma once
#include "common.h"
#include <math.h>

// Multiply-adds are written out where two kernels have to form the same number (several tokens of a request and a single one):
// which product of a sum the compiler folds into the addition is otherwise its own choice in each.
__device__ inline float rec_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

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

// The gate of normed read-outs: act(gate[t, off + i]), act 0 silu, 1 sigmoid; first: it multiplies what is normed, not the result.
struct HeadGate {
    const void *p;
    int dtype, stride, off, act, first;
    __device__ float at(size_t t, int i) const {
        if (!p) return 1.f;
        const float g = rec_ld(p, dtype, t * stride + off + i);
        return act == 1 ? rec_sigmoid(g) : rec_silu(g);
    }
};

// 8 neighbouring elements at a multiple of 16 bytes
__device__ inline void hng_ld8(const void *p, int dtype, size_t i, float (&f)[8]) {
    if (dtype == KVA_BF16) {
        const uint4 v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(p) + i);
        const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f[2 * j] = __uint_as_float(u[j] << 16);
            f[2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u);
        }
    } else {
        const float4 a = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p) + i);
        const float4 b = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p) + i + 4);
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    }
}

// The chunks of 64 tokens (recurrent_chunks.hip) of all entries of `shortest` tokens and more are numbered through.
#define REC_CHUNK_TOKENS 64

__device__ inline int rec_chunks_of(const int *__restrict__ entry_q_start, int e, int shortest) {
    const int n = entry_q_start[e + 1] - entry_q_start[e];
    return n >= shortest ? (n + REC_CHUNK_TOKENS - 1) / REC_CHUNK_TOKENS : 0;
}

// The number of the first one of entry e.  Asked by whole wavefronts.
__device__ inline int rec_first_chunk(const int *__restrict__ entry_q_start, int e, int shortest) {
    int before = 0;
    for (int x = threadIdx.x % KVA_WAVE; x < e; x += KVA_WAVE) before += rec_chunks_of(entry_q_start, x, shortest);
#pragma unroll
    for (int o = KVA_WAVE / 2; o > 0; o >>= 1) before += __shfl_xor(before, o, KVA_WAVE);
    return before;
}

// Whether an input of (an entry's n tokens, head) is infinite or not a number, as chunk_prepare_kernel leaves it per
// chunk (from `first` on) in `odd` [chunks][heads].  Asked by whole wavefronts.
__device__ inline bool rec_odd_entry(const int *__restrict__ odd, int first, int n, int heads, int head) {
    const int chunks = (n + REC_CHUNK_TOKENS - 1) / REC_CHUNK_TOKENS;
    int seen = 0;
    for (int c = threadIdx.x % KVA_WAVE; c < chunks; c += KVA_WAVE) seen |= odd[(size_t)(first + c) * heads + head];
    return __ballot(seen != 0) != 0;
}
