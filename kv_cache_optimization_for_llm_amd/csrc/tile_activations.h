// silu and erf-gelu of 32-bit sums for the products in gemm_tiles.hip and moe_tiles.hip, whose workgroup of 256 x 256 outputs has nothing
// else to do while it takes 64 to 128 of them a lane: no call of a library function, no branch, and no larger an error than expf with
// a division and erff have (common.h, moe.hip).  Against 64 bits over 16 million numbers a range, largest relative error here / there:
//   silu  z of -88 to -20 1.3e-7 / 1.6e-7, -20 to -10 1.8e-7 / 2.0e-7, -10 to 0 1.5e-7 / 1.8e-7, 0 to 20 1.2e-7 / 1.7e-7
//   gelu  z of -8 to -2 7.2e-6 / 1, -2 to -1 7.5e-7 / 1.2e-6, -1 to 0 1.2e-7 / 2.7e-7, 0 to 1.5 1.3e-7 / 1.5e-7, above 1.1e-7 / 1.1e-7
// Infinities, numbers that are none and what expf overflows for come out as there.  us: 2,048 rows of 16,384 joined outputs of 2,048 with the
// hardware's exponential of one rounded product and its reciprocal alone (errors to 3.9e-6) 100.5, this 103.2, expf and a division 108.3; the
// experts' first product, 2,048 tokens, all of 4 experts of 1,024 x 2,048, erf-gelu by one fit (5.8e-7 around 0) 42.5, this 47.2, erff 52.0.
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

// z Phi(z).  Up to |z| = 1.5: 1 + erf(z / sqrt 2) with erf as z times a polynomial in z^2 (fitted to a relative 3e-9), the polynomial's first term and
// its sum with 1 carried with their remainders, since 1 + erf cancels for negative z.  Beyond: erfc(u) = t exp(-u^2 + P(t)), t = 1 / (1 + u / 2), a
// form from Press et al., Numerical Recipes, with P fitted for u up to 10 (2e-7).
__device__ __forceinline__ float tile_gelu(float z) {
#pragma clang fp contract(off)
    const float h = 0.5f * z, s = z * z;
    float q = 8.230724120039667e-07f;
    q = fmaf(q, s, -1.7436359485145658e-05f);
    q = fmaf(q, s, 0.00022871220426168293f);
    q = fmaf(q, s, -0.002372976392507553f);
    q = fmaf(q, s, 0.01994648203253746f);
    q = fmaf(q, s, -0.13298067450523376f);
    q = fmaf(q, s, -2.4798632e-08f);
    const float a = 0.7978845834732056f * z, b = 1.f + a;
    const float rest = fmaf(z, q, fmaf(z, 0.7978845834732056f, -a)) + (a - (b - 1.f));
    const float near = fmaf(h, rest, h * b);
    const float u = fabsf(z) * 0.70710678f, t = __builtin_amdgcn_rcpf(fmaf(0.5f, u, 1.f));
    float p = 0.3398374319076538f;
    p = fmaf(p, t, -0.6068000793457031f);
    p = fmaf(p, t, 0.008121739141643047f);
    p = fmaf(p, t, 0.10939989238977432f);
    p = fmaf(p, t, 0.5368958115577698f);
    p = fmaf(p, t, 1.4437408447265625f);
    p = fmaf(p, t, -1.8258185386657715f);
    const float c = __builtin_amdgcn_exp2f(fmaf(-1.44269504f * u, u, p)), far = h * (z > 0.f ? fmaf(-t, c, 2.f) : t * c);
    // (chosen by bits: as a choice of numbers 50 us instead of 47)
    const uint32_t in = (uint32_t)((int)__float_as_uint(fabsf(z)) - (int)__float_as_uint(1.5f) >> 31);
    return __uint_as_float((__float_as_uint(near) & in) | (__float_as_uint(far) & ~in));
}
