// tp_fp64.h -- FP64 exp, exp10, log, log1p and reciprocal of the z-node arithmetic on gfx950.
//
// A node of the Limber sums is ~18 exp, ~3 log and ~8 reciprocals per point, and the device library's forms
// of them are most of its instructions.  Measured on one MI355X in units of one v_fma_f64 issue (2.03 ns per
// wave and SIMD; 8 independent chains per thread, 8192 waves):
//     exp 20, log 74, log1p 104, pow 161, x / y 13    (device library, compiler's IEEE division)
//     tp_fp64_exp 14, tp_fp64_log 18, tp_fp64_rcp 6    (here)
// What is left out is what the node arithmetic never needs: a second word of the logarithm (every one feeds an
// exponent or a sum whose own rounding is larger), the exactly rounded quotient, and branches for arguments outside the
// range.  Domain: exp takes any finite argument up to 2^30 in magnitude (it overflows to +inf and underflows to 0 there
// like the library's; a NaN stays a NaN; beyond 2^31 ln 2 = 1.49e9 the exponent's word wraps), exp10 up to 2^28, log any
// positive normal one (a zero, a denormal, an infinity or a NaN gives some finite number: where one can arrive, another
// factor of the same value carries it on), rcp any normal number whose reciprocal is normal.  The forms named _any and
// _low take what these leave out, for the places it can reach.  Errors against 80-bit arithmetic, on the device and in a
// host build alike: exp 0.91 ulp, exp10 1.19, rcp 0.50, log 0.50 ulp + 2^-60
// (tests/test_fp64_math.py).  The logarithm's table is there because its other form, 2 atanh((m - 1) / (m + 1)) with a
// reciprocal and a degree-15 series, takes 31 instructions to these 15 (25 issues to 18).
//
// The coefficients of exp are the Chebyshev interpolant of (e^r - 1 - r) / r^2 on |r| <= ln 2 / 2 (degree 9), solved in
// 60-digit arithmetic and rounded, relative remainder 1.6e-17; those of log that of (ln(1 + r) - r) / r^2 on
// |r| < 0.00397 (degree 4), absolute remainder 1.4e-19.
#pragma once
#include <cmath>
#include <cstring>

#if defined(__HIP__) || defined(__HIPCC__)
#include <hip/hip_runtime.h>
#else  // a plain host compiler: the CPU test of these forms
#define __host__
#define __device__
#define __forceinline__ inline
#endif

#if defined(__HIP_DEVICE_COMPILE__)
#define TP_FP64_DEVICE 1
#endif

// e^r for |r| <= ln 2 / 2
__host__ __device__ __forceinline__ double tp_fp64_exp_r(double r)
{
    double p = 0x1.af38a9b0ec855p-26;
    p = fma(p, r, 0x1.289185613a3d6p-22);
    p = fma(p, r, 0x1.71de0dae63bb3p-19);
    p = fma(p, r, 0x1.a019b90d2ae7ap-16);
    p = fma(p, r, 0x1.a01a01a7c41d5p-13);
    p = fma(p, r, 0x1.6c16c1788bd90p-10);
    p = fma(p, r, 0x1.11111111109b3p-7);
    p = fma(p, r, 0x1.5555555553d63p-5);
    p = fma(p, r, 0x1.5555555555556p-3);
    p = fma(p, r, 0x1.0000000000001p-1);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return p;
}

// v 2^n for t = 1.5 2^52 + n
__host__ __device__ __forceinline__ double tp_fp64_scale(double v, double t)
{
#ifdef TP_FP64_DEVICE
    return __builtin_amdgcn_ldexp(v, __double2loint(t));
#else
    long long b;
    std::memcpy(&b, &t, 8);
    return std::ldexp(v, (int)(b & 0xffffffffLL));
#endif
}

// |x| < 2^31: x = n ln 2 + r, e^x = 2^n e^r; n by the rounding of an addition to 1.5 2^52, whose low word is n
__host__ __device__ __forceinline__ double tp_fp64_exp(double x)
{
    const double t = fma(x, 0x1.71547652b82fep+0, 0x1.8p52);
    const double n = t - 0x1.8p52;
    double r = fma(n, -0x1.62e42fefa39efp-1, x);
    r = fma(n, -0x1.abc9e3b39803fp-56, r);
    return tp_fp64_scale(tp_fp64_exp_r(r), t);
}

// the same for an argument of any size, infinities among them (but a NaN gives a number: a caller has another factor
// that carries it on), and for one of any size below zero
__host__ __device__ __forceinline__ double tp_fp64_exp_low(double x) { return tp_fp64_exp(__builtin_fmax(x, -0x1p30)); }
__host__ __device__ __forceinline__ double tp_fp64_exp_any(double x) { return tp_fp64_exp_low(__builtin_fmin(x, 0x1p30)); }

// hardware reciprocal (specified to 2^29 ulp: 2^-24) and one third-order step: error e^3 = 2^-72 and the last rounding
__host__ __device__ __forceinline__ double tp_fp64_rcp_seed(double x)
{
#ifdef TP_FP64_DEVICE
    return __builtin_amdgcn_rcp(x);
#else
    return (1.0 / x) * (1.0 + 0x1p-24);  // an approximation of no more than the specified accuracy
#endif
}
__host__ __device__ __forceinline__ double tp_fp64_rcp(double x)
{
    const double r = tp_fp64_rcp_seed(x), e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}
// the same with 1 / +-infinity = +-0: there the seed is 0 and the residual a NaN, which the bound makes -1 and the step
// then 0; elsewhere the residual is far above -1
__host__ __device__ __forceinline__ double tp_fp64_rcp_any(double x)
{
    const double r = tp_fp64_rcp_seed(x), e = __builtin_fmax(fma(-x, r, 1.0), -1.0);
    return fma(r, fma(e, e, e), r);
}

// {c, -ln c} per interval of the mantissa (see the table's head); read per lane, 2 KB that stay in the vector L1
#if defined(__HIP__) || defined(__HIPCC__)
static __device__ const double tp_fp64_logtab[128][2] = {
#include "tp_fp64_logtab.inc"
};
#endif
#ifndef TP_FP64_DEVICE
static const double tp_fp64_logtab_host[128][2] = {
#include "tp_fp64_logtab.inc"
};
#endif

// ln x = k ln 2 - ln c + ln(1 + r), x = 2^k m, r = m c - 1, |r| < 0.004: with ln 2 and -ln c on multiples of 2^-43 the
// first two add exactly; the rest is a degree-6 sum.  Absolute error half an ulp of the result + 2^-60 (near x = 1 that
// is absolute, not relative: a caller that needs ln(1 + x) of a small x to its last bit does not use this).
__host__ __device__ __forceinline__ double tp_fp64_log(double x)
{
#ifdef TP_FP64_DEVICE
    const unsigned hi = (unsigned)__double2hiint(x);
    const double k = __hiloint2double(0x43300000, (int)(hi >> 20)) - (0x1p52 + 1023.0);
    const double m = __hiloint2double((int)((hi & 0xfffffu) | 0x3ff00000u), __double2loint(x));
    const double *t = tp_fp64_logtab[(hi >> 13) & 127u];
#else
    unsigned long long b;
    std::memcpy(&b, &x, 8);
    const double k = (double)(b >> 52) - 1023.0;
    const unsigned long long mb = (b & 0xfffffffffffffULL) | 0x3ff0000000000000ULL;
    double m;
    std::memcpy(&m, &mb, 8);
    const double *t = tp_fp64_logtab_host[(b >> 45) & 127u];
#endif
    const double r = fma(m, t[0], -1.0);
    double p = fma(r, -0x1.55569fde167adp-3, 0x1.999b135a6dab0p-3);
    p = fma(p, r, -0x1.ffffffffaaa5ap-3);
    p = fma(p, r, 0x1.55555555248f7p-2);
    p = fma(p, r, -0.5);
    const double q = fma(k, 0x1.ef35793c76730p-45, fma(r * r, p, r));
    return fma(k, 0x1.62e42fefa3800p-1, t[1]) + q;
}

// ln(1 + x) for x >= 0 with the same absolute error: ln u, u = 1 + x rounded, plus the rounding's share
// (x - (u - 1)) / u
__host__ __device__ __forceinline__ double tp_fp64_log1p(double x)
{
    const double u = 1.0 + x;
    const double c = u > 2.0 ? 1.0 - (u - x) : x - (u - 1.0);
#ifdef TP_FP64_DEVICE
    const double r = __builtin_amdgcn_rcp(u);
#else
    const double r = 1.0 / u;
#endif
    return tp_fp64_log(u) + c * r;
}

// 10^x, |x| < 2^28: x = n log10 2 + r, the remainder taken in decades, so that the product by ln 10 rounds a small
// number
__host__ __device__ __forceinline__ double tp_fp64_exp10(double x)
{
    const double t = fma(x, 0x1.a934f0979a371p+1, 0x1.8p52);
    const double n = t - 0x1.8p52;
    double r = fma(n, -0x1.34413509f79ffp-2, x);
    r = fma(n, 0x1.9dc1da994fd21p-59, r);
    return tp_fp64_scale(tp_fp64_exp_r(r * 0x1.26bb1bbb55516p+1), t);
}
