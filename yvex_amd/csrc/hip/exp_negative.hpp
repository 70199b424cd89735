// The exponential of the SwiGLU product's path in double. Plain arithmetic and the C library's fma, rint, fmax and ldexp,
// which are exact: a host compiler makes the same values of it.
#pragma once

#include <math.h>

namespace yvex {

// exp(x) for x <= 0: x = n ln 2 + r + c with ln 2 in two parts (Cody and Waite), the Taylor polynomial of degree 14 in
// |r| <= 0.347, whose remainder is below 2^-61, and 1 + r carried without rounding. 0.60 units in the last place at most over
// 20 million arguments against extended precision. The coefficients are loaded where they are used: those of the library's
// exponential are constants that the compiler keeps in two dozen registers around the loops of the kernel that calls it, for
// a path that one value in five hundred takes, and the registers they displace sat in scratch memory: the end of every
// chunk of a fused sweep waited for scratch loads, and with them for the weight rows asked for ahead.
__device__ const double k_exp_terms[13] = {1.0 / 87178291200.0, 1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0,
                                           1.0 / 3628800.0,     1.0 / 362880.0,     1.0 / 40320.0,     1.0 / 5040.0,
                                           1.0 / 720.0,         1.0 / 120.0,        1.0 / 24.0,        1.0 / 6.0, 0.5};
__device__ __forceinline__ double exp_of_negative(double x)
{
    const double *terms = k_exp_terms;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(terms));                              // (not known outside this path)
#endif
    x = fmax(x, -800.0);                                         // (0 from -745.2 on)
    const double n = rint(x * 0x1.71547652b82fep+0);
    const double a = fma(n, -0x1.62e42fefa3800p-1, x), b = n * 0x1.ef35793c76730p-45;
    const double r = a - b, c = (a - r) - b;
    double q = terms[0];
#pragma unroll
    for (unsigned i = 1; i < 13u; ++i) q = fma(q, r, terms[i]);
    const double h = 1.0 + r, low = (1.0 - h) + r;
    return ldexp(h + (low + fma(r * r, q, c * h)), (int)n);
}

}  // namespace yvex
