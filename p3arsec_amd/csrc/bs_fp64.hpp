// bs_fp64.hpp -- FP64 primitives for arguments known to be ordinary numbers,
// without the special-value handling of the general ones: quotients from
// v_rcp_f64 and square roots from v_rsq_f64 (relative errors at most 4.6e-8 and
// 5.3e-8, measured on random numbers of every binade of [2^-1000, 2^1000] and
// [2^-500, 2^500]), exponentials and logarithms from polynomials interpolated at
// Chebyshev nodes.  Every FMA is written out.  Largest and mean errors in units
// in the last place, measured, and of the general form each replaces:
//   quot_pos, recip_pos, sqrt_pos  0.500, 0.250   IEEE, recip64  0.500, 0.250
//   log_pos   0.87, 0.251   log64  1.18, 0.263
//   exp_mid   0.87, 0.256   the device library's exp  0.87, 0.256
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bs {

// 1 / b within half an ulp and 2^-19 of one, for |b| in [2^-1000, 2^1000]:
// with e = 1 - b y the error of the hardware's y, y (1 + e + e^2); e^3 is left
// out, below 2^-72.
__device__ __forceinline__ double recip_pos(double b) {
#pragma clang fp contract(off)
    const double y = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, y, 1.0);
    return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// a / b within an ulp: a y (1 + e + e^2), an instruction fewer than quot_pos.
__device__ __forceinline__ double quot_near(double a, double b) {
#pragma clang fp contract(off)
    const double y = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, y, 1.0);
    const double q = a * y;
    return __builtin_fma(q, __builtin_fma(e, e, e), q);
}

// a / b within half an ulp and 2^-40 of one: y to 2^-48, the quotient and its
// residual (exact in an FMA).
__device__ __forceinline__ double quot_pos(double a, double b) {
#pragma clang fp contract(off)
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

// sqrt(x), as near, for x in [2^-500, 2^500]: g and h near sqrt(x) and half its
// reciprocal, one coupled Newton step, then the residual of g.
__device__ __forceinline__ double sqrt_pos(double x) {
#pragma clang fp contract(off)
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// A positive normal x = 2^e m with m in [sqrt(1/2), sqrt(2)) (the exponent field
// counted from the high word of sqrt(1/2), as the logarithms of Sun's fdlibm do)
// and log m = f + t with f = m - 1: s = (m - 1) / (m + 1), log m = 2 atanh(s) =
// f - f^2/2 + s (f^2/2 + s^2 p(s^2)) with p = (2 atanh(s) / s - 2) / s^2
// interpolated (degree 6, relative error 5e-18).
struct LogParts {
    double e, f, t;
};
__device__ __forceinline__ LogParts log_parts(double x) {
#pragma clang fp contract(off)
    constexpr uint32_t kRootHalf = 0x3fe6a09eu;
    const uint32_t b = (uint32_t)__double2hiint(x) - kRootHalf;
    const double m = __hiloint2double((int)((b & 0xfffffu) + kRootHalf), __double2loint(x));
    const double f = m - 1.0;
    const double s = quot_near(f, m + 1.0);
    const double z = s * s;
    double p = 0.14616449685043406;
    p = __builtin_fma(p, z, 0.15331721600556042);
    p = __builtin_fma(p, z, 0.18182889125261723);
    p = __builtin_fma(p, z, 0.2222221113479508);
    p = __builtin_fma(p, z, 0.28571428625975487);
    p = __builtin_fma(p, z, 0.39999999999899505);
    p = __builtin_fma(p, z, 0.666666666666667);
    const double h = 0.5 * (f * f);
    return {(double)((int)b >> 20), f, __builtin_fma(s, __builtin_fma(z, p, h), -h)};
}
// ln 2 = kLn2Hi + kLn2Lo; kLn2Hi keeps 32 significant bits, so e kLn2Hi is exact
// for every binary exponent e of a double.
constexpr double kLn2Hi = 0.6931471803691238;        // 0x3fe62e42fee00000
constexpr double kLn2Lo = 1.9082149292705877e-10;

// log(x) of a positive normal x.  The rounding of e ln 2 + f is carried over, which
// costs three instructions and takes the largest error from 1.21 ulp to 0.87.
__device__ __forceinline__ double log_pos(double x) {
#pragma clang fp contract(off)
    const LogParts q = log_parts(x);
    const double sum = __builtin_fma(q.e, kLn2Hi, q.f);
    const double err = q.f - __builtin_fma(-q.e, kLn2Hi, sum);   // exact: |f| < ln 2, or e = 0
    return sum + (__builtin_fma(q.e, kLn2Lo, q.t) + err);
}

// The same within 1.25 ulp.
__device__ __forceinline__ double log_near(double x) {
#pragma clang fp contract(off)
    const LogParts q = log_parts(x);
    return __builtin_fma(q.e, kLn2Hi, __builtin_fma(q.e, kLn2Lo, q.f + q.t));
}

// 2^x for |x| < 1000: (2^f - 1) / f over |f| <= 1/2 (degree 10, relative error
// of 2^f 2e-17 with rounded coefficients).
__device__ __forceinline__ double exp2_mid(double x) {
#pragma clang fp contract(off)
    const double k = __builtin_rint(x);
    const double f = x - k;
    double p = 4.4549605981865186e-10;
    p = __builtin_fma(p, f, 7.072585949269223e-09);
    p = __builtin_fma(p, f, 1.0178062445845774e-07);
    p = __builtin_fma(p, f, 1.321544258792169e-06);
    p = __builtin_fma(p, f, 1.525273382983612e-05);
    p = __builtin_fma(p, f, 0.0001540353044173605);
    p = __builtin_fma(p, f, 0.0013333558146416936);
    p = __builtin_fma(p, f, 0.009618129107606888);
    p = __builtin_fma(p, f, 0.0555041086648216);
    p = __builtin_fma(p, f, 0.24022650695910097);
    p = __builtin_fma(p, f, 0.6931471805599453);
    p = __builtin_fma(p, f, 1.0);
    return __builtin_amdgcn_ldexp(p, (int)k);
}

// e^x for |x| < 1000 (0 or a subnormal below -708): x - k ln 2 with ln 2 in two
// parts, (e^f - 1) / f over |f| <= ln(2) / 2 (degree 11, relative error 7e-19;
// with degree 10, 1e-17, errors reach 0.89 ulp).
__device__ __forceinline__ double exp_mid(double x) {
#pragma clang fp contract(off)
    const double k = __builtin_rint(x * 1.4426950408889634);
    const double f = __builtin_fma(k, -kLn2Lo, __builtin_fma(k, -kLn2Hi, x));
    double p = 2.0918129454967065e-09;
    p = __builtin_fma(p, f, 2.5110037605963777e-08);
    p = __builtin_fma(p, f, 2.7557263301474753e-07);
    p = __builtin_fma(p, f, 2.755724091857897e-06);
    p = __builtin_fma(p, f, 2.4801587336421321e-05);
    p = __builtin_fma(p, f, 0.00019841269890047113);
    p = __builtin_fma(p, f, 0.0013888888888879082);
    p = __builtin_fma(p, f, 0.0083333333333196011);
    p = __builtin_fma(p, f, 0.041666666666666678);
    p = __builtin_fma(p, f, 0.1666666666666668);
    p = __builtin_fma(p, f, 0.5);
    p = __builtin_fma(p, f, 1.0);
    p = __builtin_fma(p, f, 1.0);
    return __builtin_amdgcn_ldexp(p, (int)k);
}

}  // namespace bs
