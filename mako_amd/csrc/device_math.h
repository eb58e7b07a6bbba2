// Device arithmetic that must match the host toolchain bit for bit.
// Compiled with -ffp-contract=off, IEEE fp32 division and subnormals enabled:
// every operator below rounds once, and only the explicit fma() calls fuse.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "exp_form.h"

namespace mako {

// 2^(i/32) table of glibc 2.35 (sysdeps/ieee754/flt-32/e_exp2f_data.c):
// bits(2^(i/32)) - (i << 47).
__device__ const uint64_t k_exp2_tab[32] = {
    0x3ff0000000000000, 0x3fefd9b0d3158574, 0x3fefb5586cf9890f, 0x3fef9301d0125b51,
    0x3fef72b83c7d517b, 0x3fef54873168b9aa, 0x3fef387a6e756238, 0x3fef1e9df51fdee1,
    0x3fef06fe0a31b715, 0x3feef1a7373aa9cb, 0x3feedea64c123422, 0x3feece086061892d,
    0x3feebfdad5362a27, 0x3feeb42b569d4f82, 0x3feeab07dd485429, 0x3feea47eb03a5585,
    0x3feea09e667f3bcd, 0x3fee9f75e8ec5f74, 0x3feea11473eb0187, 0x3feea589994cce13,
    0x3feeace5422aa0db, 0x3feeb737b0cdc5e5, 0x3feec49182a3f090, 0x3feed503b23e255d,
    0x3feee89f995ad3ad, 0x3feeff76f2fb5e47, 0x3fef199bdd85529c, 0x3fef3720dcef9069,
    0x3fef5818dcfba487, 0x3fef7c97337b9b5f, 0x3fefa4afa2a490da, 0x3fefd0765b6e4540,
};

// expf of glibc 2.35 as built for x86-64 with FMA, which is what std::exp(float)
// (src/gen/sampler.cpp:33) resolves to on the host: fp64 range reduction with a
// 32-entry table and a cubic, both multiply-adds of the reduction fused.
// `tab` points at k_exp2_tab or a copy of it in LDS.
// glibc leaves early for infinities and for results beyond a float.  Here such an argument is moved to a bound whose result
// the conversion at the end rounds to the same value, infinity, the least subnormal or zero (all 2^32 arguments compared), and
// nothing branches: with a branch per special case every call waited for its own table entry and its own chain, with none the
// four calls side by side overlap (the second pass over 256 rows of 151 552
// logits 123 -> 114 us, the weights of 64 rows in token order 19.7 -> 17.9).
// (exp_moved(): NaN is moved to the lower bound.)
__device__ __forceinline__ float exp_moved(float x, const uint64_t* tab)
{
    return exp_form(__builtin_amdgcn_fmed3f(x, kExpLow, kExpHigh), tab);
}
__device__ __forceinline__ float expf_glibc(float x, const uint64_t* tab)
{
    return x == x ? exp_moved(x, tab) : x + x;
}

// The three penalties of src/gen/sampler.cpp:25-27 for a token seen n times.
__device__ __forceinline__ float penalize(float l, uint32_t n, float rep, float presence, float frequency)
{
    if (rep != 1.0f)
        l = l > 0.0f ? l / rep : l * rep;
    const float fr = frequency * (float)n;
    const float dec = presence + fr;
    return l - dec;
}

// q = exp((w - m) * inv_t), src/gen/sampler.cpp:33: subtract, multiply, expf.  (0 where that is NaN: neither is a candidate,
// src/gen/sampler.cpp:34.)
__device__ __forceinline__ float weight_of(float w, float m, float inv_t, const uint64_t* tab)
{
    const float diff = w - m;
    const float x = diff * inv_t;
    return exp_moved(x, tab);
}

} // namespace mako
