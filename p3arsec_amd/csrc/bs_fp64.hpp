// bs_fp64.hpp -- FP64 primitives for arguments known to be ordinary numbers,
// without the special-value handling of the general ones: quotients from
// v_rcp_f64 (relative error at most 2^-24.3, measured over [0.007, 300]),
// square roots from v_rsq_f64, exponentials and logarithms from polynomials
// interpolated at Chebyshev nodes.  Every FMA is written out.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bs {

// 1 / b within half an ulp and 2^-24 of one, for |b| in [2^-1000, 2^1000]:
// with e = 1 - b y the error of the hardware's y, y (1 + e + e^2).
__device__ __forceinline__ double recip_pos(double b) {
#pragma clang fp contract(off)
    const double y = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, y, 1.0);
    return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// a / b within an ulp: a y (1 + e + e^2).
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

// sqrt(x) for x in [2^-500, 2^500]: g and h near sqrt(x) and half its
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

// log(x) of a positive normal x: x = 2^e m, m in [sqrt(1/2), sqrt(2)) (the
// exponent field counted from the high word of sqrt(1/2)), s = (m - 1) / (m + 1),
// log m = 2 atanh(s) with (2 atanh(s) / s - 2) / s^2 interpolated in s^2
// (degree 6, relative error 5e-18).
__device__ __forceinline__ double log_pos(double x) {
#pragma clang fp contract(off)
    constexpr uint32_t kRootHalf = 0x3fe6a09eu;
    const uint32_t b = (uint32_t)__double2hiint(x) - kRootHalf;
    const int e = (int)b >> 20;
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
    const double lm = f + __builtin_fma(s, __builtin_fma(z, p, h), -h);
    const double ed = (double)e;
    // ln 2 in two parts, the first with 32 significant bits
    return __builtin_fma(ed, 0.6931471803691238, __builtin_fma(ed, 1.9082149292705877e-10, lm));
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
// parts, (e^f - 1) / f over |f| <= ln(2) / 2 (degree 10, relative error 1e-17).
__device__ __forceinline__ double exp_mid(double x) {
#pragma clang fp contract(off)
    const double k = __builtin_rint(x * 1.4426950408889634);
    const double f = __builtin_fma(k, -1.9082149292705877e-10,
                                   __builtin_fma(k, -0.6931471803691238, x));
    double p = 2.510520638458724e-08;
    p = __builtin_fma(p, f, 2.762635725527078e-07);
    p = __builtin_fma(p, f, 2.7557255425720897e-06);
    p = __builtin_fma(p, f, 2.480150434696448e-05);
    p = __builtin_fma(p, f, 0.00019841269874800512);
    p = __builtin_fma(p, f, 0.0013888888932488625);
    p = __builtin_fma(p, f, 0.008333333333326141);
    p = __builtin_fma(p, f, 0.04166666666657314);
    p = __builtin_fma(p, f, 0.1666666666666667);
    p = __builtin_fma(p, f, 0.5000000000000006);
    p = __builtin_fma(p, f, 1.0);
    p = __builtin_fma(p, f, 1.0);
    return __builtin_amdgcn_ldexp(p, (int)k);
}

}  // namespace bs
