/*
 * p2m_fast64.h -- double-precision device functions for values (not for
 * decisions that must agree bit for bit with the reference: those use
 * p2m_math.h): fused multiply-adds, refined hardware reciprocals, arguments
 * taken to be normal numbers in the ranges stated.
 */
#ifndef P2M_FAST64_H
#define P2M_FAST64_H

#include "p2m_math.h"

/* square root, ln x and e^x of normal arguments (x > 0 for the first two):
 * a refined reciprocal square root, and the series of p2m_log and p2m_exp with
 * fused multiply-adds and the quotient by a refined reciprocal; a few 1e-16
 * relative, as those */
__device__ static inline double f64_sqrt(double x)
{
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

__device__ static inline double f64_log(double x)
{
    double m = __builtin_amdgcn_frexp_mant(x);
    int e = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0x1.6a09e667f3bcdp-1;
    m = low ? 2.0 * m : m;
    e = low ? e - 1 : e;
    const double d = m + 1.0, nn = m - 1.0;
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
    double s = nn * r;
    s = __builtin_fma(r, __builtin_fma(-s, d, nn), s);
    const double z = s * s;
    double p = 0x1.642c8590b2164p-4;
    p = __builtin_fma(z, p, 0x1.8618618618618p-4);
    p = __builtin_fma(z, p, 0x1.af286bca1af28p-4);
    p = __builtin_fma(z, p, 0x1.e1e1e1e1e1e1ep-4);
    p = __builtin_fma(z, p, 0x1.1111111111111p-3);
    p = __builtin_fma(z, p, 0x1.3b13b13b13b14p-3);
    p = __builtin_fma(z, p, 0x1.745d1745d1746p-3);
    p = __builtin_fma(z, p, 0x1.c71c71c71c71cp-3);
    p = __builtin_fma(z, p, 0x1.2492492492492p-2);
    p = __builtin_fma(z, p, 0x1.999999999999ap-2);
    p = __builtin_fma(z, p, 0x1.5555555555555p-1);
    const double k = (double)e;
    return __builtin_fma(k, P2M_LN2_HI, __builtin_fma(k, P2M_LN2_LO, __builtin_fma(s * z, p, 2.0 * s)));
}

__device__ static inline double f64_exp(double x)
{
    const double k = __builtin_rint(x * P2M_INVLN2);
    double r = __builtin_fma(-k, P2M_LN2_HI, x);
    r = __builtin_fma(-k, P2M_LN2_LO, r);
    double p = 0x1.6124613a86d09p-33;
    p = __builtin_fma(r, p, 0x1.1eed8eff8d898p-29);
    p = __builtin_fma(r, p, 0x1.ae64567f544e4p-26);
    p = __builtin_fma(r, p, 0x1.27e4fb7789f5cp-22);
    p = __builtin_fma(r, p, 0x1.71de3a556c734p-19);
    p = __builtin_fma(r, p, 0x1.a01a01a01a01ap-16);
    p = __builtin_fma(r, p, 0x1.a01a01a01a01ap-13);
    p = __builtin_fma(r, p, 0x1.6c16c16c16c17p-10);
    p = __builtin_fma(r, p, 0x1.1111111111111p-7);
    p = __builtin_fma(r, p, 0x1.5555555555555p-5);
    p = __builtin_fma(r, p, 0x1.5555555555555p-3);
    p = __builtin_fma(r, p, 0.5);
    return __builtin_amdgcn_ldexp(1.0 + __builtin_fma(r * r, p, r), (int)k);
}

/* ln tan(theta) - ln(q) / 2 for small angles (theta below 0.11), by its series
 * in q (the next term is below 1e-17): q = sin^2(theta), and q = theta^2 */
__device__ static inline double f64_lntan_sin2(double q)
{
    double p = __builtin_fma(q, 1.0 / 16.0, 1.0 / 14.0);
    p = __builtin_fma(q, p, 1.0 / 12.0);
    p = __builtin_fma(q, p, 1.0 / 10.0);
    p = __builtin_fma(q, p, 1.0 / 8.0);
    p = __builtin_fma(q, p, 1.0 / 6.0);
    p = __builtin_fma(q, p, 1.0 / 4.0);
    p = __builtin_fma(q, p, 1.0 / 2.0);
    return q * p;
}
__device__ static inline double f64_lntan_angle(double q)
{
    double p = __builtin_fma(q, 0x1.0d071e8bccf11p-12, 0x1.83256720c7d4ep-11);
    p = __builtin_fma(q, p, 0x1.1e5e18380dc2bp-9);
    p = __builtin_fma(q, p, 0x1.b85fca40e852dp-8);
    p = __builtin_fma(q, p, 0x1.664f4882c10fap-6);
    p = __builtin_fma(q, p, 0x1.3e93e93e93e94p-4);
    p = __builtin_fma(q, p, 0x1.5555555555555p-2);
    return q * p;
}
#define F64_SMALL_Q 0.0121       /* q up to here */

#endif
