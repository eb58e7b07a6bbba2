// The kernels' expf behind the bounds of its argument: plain C++ so that the host test of every argument and the HIP kernels share
// one implementation (compiled with -ffp-contract=off: only the explicit multiply-adds fuse).
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define EXPFORM_HD __host__ __device__ __forceinline__
#else
#define EXPFORM_HD inline
#endif

namespace mako {

// Arguments are moved to between these, whose results round to zero (or the least subnormal) and to infinity.
constexpr float kExpLow = -104.0f, kExpHigh = 89.0f;

// e^x for kExpLow <= x <= kExpHigh; `tab`: bits(2^(i/32)) - (i << 47).
// The cubic by Horner's rule, scaled in its last multiply-add: an operation fewer than glibc's order, and the same float for
// every argument (tests/cpu/exp_core_test.cpp).  With the scale put together as two words the kernels, bound by vector instructions,
// have five fewer a weight: the weights of 64 rows of 129 280 logits in token order 18.7 -> 16.9 us, the second pass over 512 rows
// 57 -> 55.
EXPFORM_HD float exp_form(float x, const uint64_t* tab)
{
    const double inv_ln2_n = 0x1.71547652b82fep+0 * 32.0;
    const double shift = 0x1.8p+52;
    const double c0 = 0x1.c6af84b912394p-5 / 32 / 32 / 32;
    const double c1 = 0x1.ebfce50fac4f3p-3 / 32 / 32;
    const double c2 = 0x1.62e42ff0c52d6p-1 / 32;
    const double xd = (double)x;
    double kd = __builtin_fma(inv_ln2_n, xd, shift);
    const uint32_t ki = (uint32_t)__builtin_bit_cast(uint64_t, kd);
    kd -= shift;
    const double r = __builtin_fma(inv_ln2_n, xd, -kd);
    // (+ ki << 47, which the lower word has no part in.  As two words to the end: of a 64-bit sum the compiler makes five instructions)
    typedef uint32_t words __attribute__((vector_size(8)));
    words t = __builtin_bit_cast(words, tab[ki & 31u]);
    t[1] += ki << 15;
    const double s = __builtin_bit_cast(double, t);
    return (float)__builtin_fma(__builtin_fma(r, __builtin_fma(c0, r, c1), c2), r * s, s);
}

} // namespace mako
