// tp_fp64.h -- FP64 exp, exp10, log, log1p and reciprocal of the z-node arithmetic on gfx950.
//
// A node of the Limber sums is ~18 exp, ~3 log and ~8 reciprocals per point, and the device library's forms
// of them are most of its instructions.  Measured on one MI355X in units of one v_fma_f64 issue (2.03 ns per
// wave and SIMD; 8 independent chains per thread, 8192 waves):
//     exp 20, log 74, log1p 104, pow 161, x / y 13    (device library, compiler's IEEE division)
//     tp_fp64_exp 14, tp_fp64_log 25, tp_fp64_rcp 6    (here)
// What is left out is what the node arithmetic never needs: a second word of the logarithm (every one feeds an
// exponent or a sum whose own rounding is larger), the exactly rounded quotient, and branches for arguments
// outside the range.  Domain: exp takes any finite argument below 2^31 in magnitude (it overflows to +inf and
// underflows to 0 there like the library's), log any positive finite one (zeros, negative numbers and
// infinities are stopped before the node loop; a NaN stays a NaN), rcp any normal number whose reciprocal is
// normal.  Errors against 80-bit arithmetic: exp 0.91 ulp, log 0.93, log1p 1.17, exp10 1.19, rcp 0.50 (tests/test_fp64_math.py).
//
// The coefficients are Chebyshev interpolants of (e^r - 1 - r) / r^2 on |r| <= ln 2 / 2 (degree 9) and of
// 2 (atanh(s) / s - 1) / s^2 on |s| <= (sqrt 2 - 1) / (sqrt 2 + 1) (degree 6 in s^2), solved in 60-digit
// arithmetic and rounded; relative remainders 1.6e-17 and 4.6e-18.
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

// hardware reciprocal (2^-27 or better) and one third-order step: error e^3 + the last rounding
__host__ __device__ __forceinline__ double tp_fp64_rcp(double x)
{
#ifdef TP_FP64_DEVICE
    const double r = __builtin_amdgcn_rcp(x);
#else
    const double r = (1.0 / x) * (1.0 + 0x1p-27);  // an approximation of no more than the hardware's accuracy
#endif
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// k ln 2 + ln(1 + f) for 1 + f in [sqrt(1/2), sqrt(2)): with s = f / (2 + f), ln(1 + f) = 2 atanh(s) =
// f - s (f - z P(z)), z = s^2; f is exact, and the rounding of s enters weighted by |f - z P| < 0.42
__host__ __device__ __forceinline__ double tp_fp64_log_kf(double k, double f)
{
    const double s = f * tp_fp64_rcp(f + 2.0);
    const double z = s * s;
    double p = 0x1.2b5900de53b32p-3;
    p = fma(p, z, 0x1.39fe51a7c18f9p-3);
    p = fma(p, z, 0x1.7462b51cb66b1p-3);
    p = fma(p, z, 0x1.c71c62e3f11e6p-3);
    p = fma(p, z, 0x1.2492492df281ap-2);
    p = fma(p, z, 0x1.99999999952d7p-2);
    p = fma(p, z, 0x1.5555555555558p-1);
    const double q = fma(-s, fma(-z, p, f), k * 0x1.abc9e3b39803fp-56);
    return fma(k, 0x1.62e42fefa39efp-1, f + q);
}

__host__ __device__ __forceinline__ void tp_fp64_split(double x, double *m, int *k)
{
#ifdef TP_FP64_DEVICE
    *m = __builtin_amdgcn_frexp_mant(x);
    *k = __builtin_amdgcn_frexp_exp(x);
#else
    *m = std::frexp(x, k);
#endif
    const bool lo = *m < 0x1.6a09e667f3bcdp-1;
    *m = lo ? *m + *m : *m;
    *k = lo ? *k - 1 : *k;
}

__host__ __device__ __forceinline__ double tp_fp64_log(double x)
{
    double m;
    int k;
    tp_fp64_split(x, &m, &k);
    return tp_fp64_log_kf((double)k, m - 1.0);
}

// ln(1 + x) for x >= 0 (or a NaN): ln u, u = 1 + x rounded, plus the rounding's share (x - (u - 1)) / u
__host__ __device__ __forceinline__ double tp_fp64_log1p(double x)
{
    const double u = 1.0 + x;
    double m;
    int k;
    tp_fp64_split(u, &m, &k);
    const double f = m - 1.0;
    const double c = u > 2.0 ? 1.0 - (u - x) : x - (u - 1.0);
#ifdef TP_FP64_DEVICE
    const double r = __builtin_amdgcn_rcp(u);
#else
    const double r = 1.0 / u;
#endif
    return tp_fp64_log_kf((double)k, f) + c * r;
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
