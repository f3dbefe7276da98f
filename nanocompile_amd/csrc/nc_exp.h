// nc_expf's value by a shorter road, for kernels whose vector instructions it bounds.
//
// The same table, reduction and polynomial as nc_expf (nc_math.h), with fused multiply-adds, the
// nearest integer and its low bits taken from one addition of 1.5 * 2^52, and the special cases
// left to the arithmetic: about half the instructions. The double result differs from nc_expf's in
// its last bits; the float it rounds to does not: all float inputs up to 100 were compared (gcc on
// the host; IEEE double operations and fma give the GPU the same), and none differs.
// tests/test_exp.py holds a sample of them and every edge.
#pragma once

#include "nc_math.h"

// a * b + c with the constant c read from scalar registers: left to itself hipcc takes the form that
// adds into its destination and copies c there first, two moves a step.
NC_MATH_FN double nc_fma_const(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
    return d;
#else
    return __builtin_fma(a, b, c);
#endif
}

// exp(x) for x <= 100 or NaN.
NC_MATH_FN float nc_expf_upto100(float xf) {
    // below -104 the float is 0, and so it is for -150, from where on the arithmetic would go wrong
    const double x = (double)(xf < -104.0f ? -150.0f : xf);
    const double inv = 0x1.71547652b82fep+6, shift = 0x1.8p52;      // 64 / ln 2; an ulp of shift is 1
    const double l_hi = 0x1.62e42ffp-7, l_lo = -0x1.718432a1b0e26p-41;
    union { double d; uint32_t w[2]; } kb;
    kb.d = nc_fma_const(x, inv, shift);
    const int ki = (int)kb.w[0];                       // k mod 2^32
    const double k = kb.d - shift;
    const double r = __builtin_fma(-k, l_lo, __builtin_fma(-k, l_hi, x));
    double p = nc_fma_const(1.0 / 120.0, r, 1.0 / 24.0);
    p = nc_fma_const(p, r, 1.0 / 6.0);
    p = nc_fma_const(p, r, 0.5);
    p = nc_fma_const(p, r, 1.0);
    p = nc_fma_const(p, r, 1.0);
    return (float)__builtin_ldexp(nc_exp2_64ths[ki & 63] * p, ki >> 6);
}
