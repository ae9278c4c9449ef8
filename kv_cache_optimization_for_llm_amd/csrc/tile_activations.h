// silu of 32-bit sums for the products in gemm_tiles.hip and moe_tiles.hip, whose workgroup of 256 x 256 outputs has nothing else to do
// while it takes 64 of them a lane: no call of a library function, no branch, and no larger an error than expf with a division has
// (common.h).  Against 64 bits over 16 million numbers a range, largest relative error here / there: z of -88 to -20 1.3e-7 / 1.6e-7, -20 to -10
// 1.8e-7 / 2.0e-7, -10 to 0 1.5e-7 / 1.8e-7, 0 to 20 1.2e-7 / 1.7e-7.  Infinities, numbers that are none and what expf overflows for come out as
// there.  us: 2,048 rows of 16,384 joined outputs of 2,048 with the hardware's exponential of one rounded product and its reciprocal alone
// (errors to 3.9e-6) 100.5, this 103.2, expf and a division 108.3.
#pragma once
#include "common.h"

__device__ __forceinline__ float tile_silu(float z) {
#pragma clang fp contract(off)
    // e^-z as 2^n 2^f, with f off by 2^-26 whatever z is; z over 1 + e^-z, both a sixteenth so that the reciprocal is no denormal, with one
    // correction by the division's remainder
    const float t = __builtin_amdgcn_fmed3f(z, -200.f, 200.f), n = rintf(-1.44269504f * t), f = fmaf(t, -1.92596299e-8f, fmaf(t, -1.44269502f, -n));
    const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n), d = fmaf(e, 0.0625f, 0.0625f), r = __builtin_amdgcn_rcpf(d);
    const float x = 0.0625f * z, q = x * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, x), r, q), d, x);
}
