// Test-only: the FP64 primitives for ordinary numbers (p3arsec_amd/csrc/bs_fp64.hpp)
// on the GPU against the host's 64-bit-mantissa long double, in units in the last
// place of the exact result, beside the general ones they stand in for (the
// device library's exp, log64 and recip64 of bs_math.hpp, IEEE division and
// square root).  Inputs: random numbers of the ranges the map and the swaptions
// meet, every binade of the range a function states, and the neighbourhoods of
// sqrt(1/2), 1 and sqrt(2).  Moro's inverse normal (bs_moro.hpp) in the form the
// linear kernel takes and in the reference's, in absolute error.
//
//   fp64_ordinary     prints "name inputs max at mean" per function: errors in
//                     ulps, relative ones of the hardware's reciprocal and
//                     reciprocal root over every binade, absolute ones of Moro's.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <random>
#include <string>
#include <vector>

#include "bs_math.hpp"
#include "bs_moro.hpp"

#define HIP_OK(x)                                                                  \
    do {                                                                           \
        hipError_t e_ = (x);                                                       \
        if (e_ != hipSuccess) {                                                    \
            fprintf(stderr, "%s: %s\n", #x, hipGetErrorString(e_));                \
            exit(2);                                                               \
        }                                                                          \
    } while (0)

enum Fn { kQuotPos, kDiv, kRecipPos, kRecip64, kSqrtPos, kSqrt, kLogPos, kLog64, kExpMid, kExp,
          kExp2Mid, kRcp, kRsq, kMoro, kMoroRef, kLog };

__global__ void k_eval(int fn, const double* a, const double* b, double* y, int64_t n) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double x = a[i];
    switch (fn) {
        case kQuotPos: y[i] = bs::quot_pos(x, b[i]); break;
        case kDiv: y[i] = x / b[i]; break;
        case kRecipPos: y[i] = bs::recip_pos(x); break;
        case kRecip64: y[i] = bs::recip64(x); break;
        case kSqrtPos: y[i] = bs::sqrt_pos(x); break;
        case kSqrt: y[i] = ::sqrt(x); break;
        case kLogPos: y[i] = bs::log_pos(x); break;
        case kLog64: y[i] = bs::log64(x); break;
        case kExpMid: y[i] = bs::exp_mid(x); break;
        case kExp: y[i] = ::exp(x); break;
        case kExp2Mid: y[i] = bs::exp2_mid(x); break;
        case kRcp: y[i] = __builtin_amdgcn_rcp(x); break;
        case kRsq: y[i] = __builtin_amdgcn_rsq(x); break;
        case kLog: y[i] = ::log(x); break;
        case kMoro: {   // x: a residue
            const uint32_t r = (uint32_t)x;
            const bs::MoroCentral central;
            y[i] = r > bs::kTailLo && r < bs::kTailHi ? central(r) : bs::moro_tail_fma(r);
            break;
        }
        case kMoroRef: y[i] = bs::moro_inv(x * 4.656612875e-10); break;
    }
}

// Moro's inverse normal of u (Glasserman 2003, fig. 2.13).
static long double moro(long double u) {
    static const double A[] = {2.50662823884, -18.61500062529, 41.39119773534, -25.44106049637};
    static const double B[] = {-8.47351093090, 23.08336743743, -21.06224101826, 3.13082909833};
    static const double C[] = {0.3374754822726147, 0.9761690190917186, 0.1607979714918209,
                               0.0276438810333863, 0.0038405729373609, 0.0003951896511919,
                               0.0000321767881768, 0.0000002888167364, 0.0000003960315187};
    const long double x = u - 0.5L;
    auto horner = [](const double* c, int n, long double t) {
        long double v = c[n - 1];
        for (int i = n - 2; i >= 0; --i) v = v * t + c[i];
        return v;
    };
    if (fabs((double)x) < 0.42)
        return x * horner(A, 4, x * x) / (horner(B, 4, x * x) * (x * x) + 1.0L);
    const long double v = horner(C, 9, logl(-logl(x > 0 ? 1.0L - u : u)));
    return x < 0 ? -v : v;
}

static long double exact(int fn, double a, double b) {
    const long double x = a;
    switch (fn) {
        case kMoro:
        case kMoroRef: return moro(a * 4.656612875e-10);   // u as ran_unif rounds it
        case kQuotPos:
        case kDiv: return x / b;
        case kRecipPos:
        case kRecip64:
        case kRcp: return 1.0L / x;
        case kSqrtPos:
        case kSqrt: return sqrtl(x);
        case kRsq: return 1.0L / sqrtl(x);
        case kLogPos:
        case kLog:
        case kLog64: return logl(x);
        case kExpMid:
        case kExp: return expl(x);
        default: return exp2l(x);
    }
}

// The last place of a double next to r (a subnormal's at least).
static long double ulp_of(long double r) {
    int e;
    frexpl(r, &e);
    return ldexpl(1.0L, std::max(e - 53, -1074));
}

static double* da;
static double* db;
static double* dy;

static void run(const char* name, int fn, const std::vector<double>& a,
                const std::vector<double>& b, char unit = 'u') {
    const int64_t n = (int64_t)a.size();
    std::vector<double> y(n);
    HIP_OK(hipMemcpy(da, a.data(), n * sizeof(double), hipMemcpyHostToDevice));
    if (!b.empty()) HIP_OK(hipMemcpy(db, b.data(), n * sizeof(double), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_eval, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, fn, da, db, dy,
                       n);
    HIP_OK(hipGetLastError());
    HIP_OK(hipMemcpy(y.data(), dy, n * sizeof(double), hipMemcpyDeviceToHost));
    long double worst = 0, sum = 0;
    double at = 0;
    for (int64_t i = 0; i < n; ++i) {
        const long double r = exact(fn, a[i], b.empty() ? 0.0 : b[i]);
        long double e = fabsl((long double)y[i] - r) /
                        (unit == 'u' ? ulp_of(r) : unit == 'r' ? fabsl(r) : 1.0L);
        if (!(e >= 0)) e = 1e30L;   // NaN
        sum += e;
        if (e > worst) worst = e, at = a[i];
    }
    printf("%s %lld %.6Lg %a %.6Lg\n", name, (long long)n, worst, at, sum / n);
    fflush(stdout);
}

int main() {
    std::mt19937_64 rng(20261205);
    const size_t N = 1 << 21, kMost = 3 * N + 3 * 8193;
    HIP_OK(hipMalloc(&da, kMost * sizeof(double)));
    HIP_OK(hipMalloc(&db, kMost * sizeof(double)));
    HIP_OK(hipMalloc(&dy, kMost * sizeof(double)));
    auto uniform = [&](double lo, double hi, size_t n, std::vector<double>* v) {
        std::uniform_real_distribution<double> u(lo, hi);
        for (size_t i = 0; i < n; ++i) v->push_back(u(rng));
    };
    auto binades = [&](int lo, int hi, size_t n, std::vector<double>* v) {
        std::uniform_real_distribution<double> u(1.0, 2.0);
        for (size_t i = 0; i < n; ++i)
            v->push_back(ldexp(u(rng), lo + (int)(rng() % (uint64_t)(hi - lo))));
    };
    std::vector<double> none, x, y;
    uniform(1.0, 20.0, N, &x), binades(-1000, 1000, N, &x);
    run("recip_pos", kRecipPos, x, none), run("recip64", kRecip64, x, none);
    run("rcp_relative", kRcp, x, none, 'r');
    x.clear();
    uniform(10.0, 300.0, N, &x), uniform(10.0, 200.0, N, &y);      // S / K
    uniform(-3.0, 3.0, N, &x), uniform(0.007, 1.0, N, &y);         // d1
    binades(-250, 250, N, &x), binades(-250, 250, N, &y);
    run("quot_pos", kQuotPos, x, y), run("division", kDiv, x, y);
    x.clear();
    uniform(0.01, 3.0, N, &x), binades(-500, 500, N, &x);
    run("sqrt_pos", kSqrtPos, x, none), run("sqrt", kSqrt, x, none);
    run("rsq_relative", kRsq, x, none, 'r');
    x.clear();
    uniform(0.5, 2.0, N, &x), uniform(0.0, 0.08, N, &x), binades(-1022, 1023, N, &x);
    for (double c : {M_SQRT1_2, 1.0, M_SQRT2}) {
        double d = c;
        for (int k = 0; k < 4096; ++k) d = nextafter(d, 0.0);
        for (int k = 0; k <= 8192; ++k, d = nextafter(d, 4.0)) x.push_back(d);
    }
    run("log_pos", kLogPos, x, none), run("log64", kLog64, x, none), run("log", kLog, x, none);
    x.clear();
    uniform(-20.0, 0.0, N, &x), uniform(-0.3, 0.3, N, &x), uniform(-708.0, 709.0, N, &x);
    run("exp_mid", kExpMid, x, none), run("exp", kExp, x, none);
    x.clear();
    uniform(-745.0, -708.5, N, &x);
    run("exp_mid_subnormal", kExpMid, x, none);
    x.clear();
    uniform(-4.0, 4.0, N, &x), uniform(-1000.0, 1000.0, N, &x);
    run("exp2_mid", kExp2Mid, x, none);
    for (bool tail : {false, true}) {
        x.clear();
        for (size_t i = 0; i < N; ++i) {
            const uint64_t width = tail ? bs::kTailLo : bs::kTailHi - bs::kTailLo - 1;
            const uint64_t r = rng() % width + (tail ? 1 : bs::kTailLo + 1);
            x.push_back((double)(tail && i % 2 ? bs::kM31 - r : r));
        }
        run(tail ? "moro_tail" : "moro_central", kMoro, x, none, 'a');
        run(tail ? "moro_tail_reference" : "moro_central_reference", kMoroRef, x, none, 'a');
    }
    HIP_OK(hipFree(da));
    HIP_OK(hipFree(db));
    HIP_OK(hipFree(dy));
    return 0;
}
