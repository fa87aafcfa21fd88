// bs_moro.hpp -- Moro's inverse normal, as the step-by-step swaptions kernel
// evaluates it (the reference's arithmetic, statement by statement) and as the
// linear form does (from a generator's residue, with FMAs).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "bs_fp64.hpp"

namespace bs {

constexpr uint64_t kM31 = 2147483647u;   // the generator's modulus

// Moro's inverse normal (Moro 1995; Glasserman, Monte Carlo Methods in
// Financial Engineering, fig. 2.13), as PARSEC's CumNormalInv evaluates it:
// a rational function of x = u - 0.5 for |x| < 0.42, a Chebyshev series in
// log(-log(min(u, 1 - u))) outside.
__device__ __forceinline__ double moro_central(double x) {
#pragma clang fp contract(off)
    const double r = x * x;
    const double num = x * (((-25.44106049637 * r + 41.39119773534) * r + -18.61500062529) * r +
                            2.50662823884);
    const double den = (((3.13082909833 * r + -21.06224101826) * r + 23.08336743743) * r +
                        -8.47351093090) * r + 1.0;
    return num / den;
}

__device__ __forceinline__ double moro_tail(double u) {
#pragma clang fp contract(off)
    const double x = u - 0.5;
    double t = x > 0.0 ? 1.0 - u : u;
    t = log(-log(t));
    t = 0.3374754822726147 + t * (0.9761690190917186 + t * (0.1607979714918209 +
        t * (0.0276438810333863 + t * (0.0038405729373609 + t * (0.0003951896511919 +
        t * (0.0000321767881768 + t * (0.0000002888167364 + t * 0.0000003960315187)))))));
    return x < 0.0 ? -t : t;
}

__device__ __forceinline__ double moro_inv(double u) {
    const double x = u - 0.5;
    return fabs(x) < 0.42 ? moro_central(x) : moro_tail(u);
}

// Residues whose uniform |u - 0.5| >= 0.42 takes Moro's tail: x <= kTailLo or
// x >= kTailHi, u rounded as in ran_unif.
constexpr bool in_tail(uint32_t x) {
    const double d = (double)x * 4.656612875e-10 - 0.5;
    return !((d < 0 ? -d : d) < 0.42);
}
constexpr uint32_t tail_edge(bool upper) {
    uint32_t a = upper ? (uint32_t)kM31 / 2 : 0, b = upper ? (uint32_t)kM31 - 1 : (uint32_t)kM31 / 2;
    while (b - a > 1) {   // upper: b is in the tail and a is not; lower: a is and b is not
        const uint32_t c = a + (b - a) / 2;
        if (in_tail(c) == upper) b = c;
        else a = c;
    }
    return upper ? b : a;
}
constexpr uint32_t kTailLo = tail_edge(false), kTailHi = tail_edge(true);
static_assert(in_tail(kTailLo) && !in_tail(kTailLo + 1) && in_tail(kTailHi) &&
                  !in_tail(kTailHi - 1) && in_tail(0) && in_tail((uint32_t)kM31 - 1),
              "tail residues");

// A constant held in a vector register from here on.  An FP64 instruction reads
// one scalar operand at most and there are not enough scalar registers for
// every constant of k_sw_paths, so the compiler otherwise builds the central
// branch's constants anew for every draw, 6 of its 23 instructions.
__device__ __forceinline__ double pinned(double c) {
    asm("" : "+v"(c));
    return c;
}

// Moro's two branches (moro_central, moro_tail) with FMAs, from u rounded as in
// ran_unif: at the upper end, where 1 - u is small, an unrounded u moves the
// normal by up to 7.8e-11.  Largest and mean errors against 64-bit mantissas on 2M
// residues: central 2.9e-15 and 9.8e-17 (moro_central 4.3e-15 and 1.23e-16), tail
// 1.46e-15 and 1.364e-16 (moro_tail 1.72e-15 and 1.386e-16).  The rounding is one
// instruction a draw (PARSEC's native run 753 us without it, 771 with it).
struct MoroCentral {
    double scale = pinned(4.656612875e-10);
    double a1 = pinned(-25.44106049637), a2 = pinned(41.39119773534),
           a3 = pinned(-18.61500062529), a4 = pinned(2.50662823884);
    double b1 = pinned(3.13082909833), b2 = pinned(-21.06224101826),
           b3 = pinned(23.08336743743), b4 = pinned(-8.47351093090);
    // The normal of residue x's uniform, for the residues outside the tail.
    __device__ __forceinline__ double operator()(uint32_t residue) const {
#pragma clang fp contract(off)
        const double x = (double)residue * scale - 0.5;
        const double r = x * x;
        double num = __builtin_fma(r, a1, a2);
        num = __builtin_fma(r, num, a3);
        num = __builtin_fma(r, num, a4);
        double den = __builtin_fma(r, b1, b2);
        den = __builtin_fma(r, den, b3);
        den = __builtin_fma(r, den, b4);
        den = __builtin_fma(r, den, 1.0);   // 0.11 <= den <= 1 for |x| <= 0.42
        return quot_near(x * num, den);
    }
};

// The normal of a nonzero residue in the tail: log(-log(min(u, 1 - u))).
__device__ __forceinline__ double moro_tail_fma(uint32_t residue) {
#pragma clang fp contract(off)
    const bool upper = residue > (uint32_t)kM31 / 2;
    const double u = (double)residue * 4.656612875e-10;
    const double t = log_near(-log_near(upper ? 1.0 - u : u));
    double v = __builtin_fma(t, 0.0000003960315187, 0.0000002888167364);
    v = __builtin_fma(t, v, 0.0000321767881768);
    v = __builtin_fma(t, v, 0.0003951896511919);
    v = __builtin_fma(t, v, 0.0038405729373609);
    v = __builtin_fma(t, v, 0.0276438810333863);
    v = __builtin_fma(t, v, 0.1607979714918209);
    v = __builtin_fma(t, v, 0.9761690190917186);
    v = __builtin_fma(t, v, 0.3374754822726147);
    return upper ? v : -v;
}

}  // namespace bs
