// FP64 exponential and cutoff cosine of the per-entry loops, and the networks' tanh.
//
// The per-entry kernels are bound by VALU issue, and most of their instructions were the library's exp (about 30
// with the range checks and a register move per polynomial coefficient, which the compiler keeps in VGPRs) and
// sincospi (about 110 with its argument reduction).  Here each polynomial step is one v_fma_f64 with its
// coefficient in an SGPR pair, and the arguments' ranges are used: 18 instructions for e^x, about 30 for the
// cutoff's sine and cosine.  The coefficients are minimax fits (Remez exchange in 50-digit arithmetic) of the
// stated functions.
#pragma once

#include <hip/hip_runtime.h>

namespace atomnn {

// a b + c with a wave-uniform c read from SGPRs
__device__ __forceinline__ double fma_sc(double a, double b, double c) {
    double o;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(o) : "v"(a), "v"(b), "s"(c));
    return o;
}

// e^x.  x = n ln 2 + r, |r| <= ln 2 / 2; e^r = 1 + r (1 + r q(r)), q of degree 9 (fit error 3.6e-18); below -1000
// (where e^x is 0 in FP64) the argument is held, so that infinite products give 0.  On 30,000 points
// of [-100, 0] the error is at most 0.79 ulp and 0.292 ulp rms, the same as the library's.
__device__ __forceinline__ double exp_f64(double x) {
    x = x < -1000.0 ? -1000.0 : x;  // (a NaN stays one)
    const double n = rint(x * 1.4426950408889634);
    double r = fma(n, -0.6931471805599453, x);
    r = fma(n, -2.3190468138462996e-17, r);
    double q = 2.5117605919396305e-08;
    q = fma_sc(q, r, 2.7630856171049715e-07);
    q = fma_sc(q, r, 2.755721721092878e-06);
    q = fma_sc(q, r, 2.4801491260699277e-05);
    q = fma_sc(q, r, 0.00019841269916209367);
    q = fma_sc(q, r, 0.001388888894557356);
    q = fma_sc(q, r, 0.008333333333307848);
    q = fma_sc(q, r, 0.04166666666652186);
    q = fma_sc(q, r, 0.166666666666667);
    q = fma_sc(q, r, 0.5000000000000012);
    q = fma(q, r, 1.0);
    q = fma(q, r, 1.0);
    return ldexp(q, (int)n);
}

// tanh z = -m / (2 + m) with m = e^(-2|z|) - 1, sign of z.  With 2^n and r as above, m = 2^n (e^r - 1) + (2^n - 1):
// nothing cancels (n = 0 near z = 0, where m = e^r - 1 = r (1 + r q)).  The quotient's divisor lies in [1, 2], so
// the reciprocal needs no scaling: v_rcp_f64 and two Newton steps, and a correction of the product.  About 35
// instructions (expm1 and the compiler's division: about 90).
__device__ __forceinline__ double tanh_f64(double z) {
    double x = -2.0 * fabs(z);
    x = x < -1000.0 ? -1000.0 : x;  // (a NaN stays one)
    const double n = rint(x * 1.4426950408889634);
    double r = fma(n, -0.6931471805599453, x);
    r = fma(n, -2.3190468138462996e-17, r);
    double q = 2.5117605919396305e-08;
    q = fma_sc(q, r, 2.7630856171049715e-07);
    q = fma_sc(q, r, 2.755721721092878e-06);
    q = fma_sc(q, r, 2.4801491260699277e-05);
    q = fma_sc(q, r, 0.00019841269916209367);
    q = fma_sc(q, r, 0.001388888894557356);
    q = fma_sc(q, r, 0.008333333333307848);
    q = fma_sc(q, r, 0.04166666666652186);
    q = fma_sc(q, r, 0.166666666666667);
    q = fma_sc(q, r, 0.5000000000000012);
    const double p = fma(r * r, q, r);  // e^r - 1
    const double s = ldexp(1.0, (int)n), m = fma(s, p, s - 1.0), d = 2.0 + m;
    double y = __builtin_amdgcn_rcp(d);
    y = fma(fma(-d, y, 1.0), y, y);
    y = fma(fma(-d, y, 1.0), y, y);
    double t = -m * y;
    t = fma(fma(-d, t, -m), y, t);
    return copysign(t, z);
}

// sin(pi x) and cos(pi x) for 0 <= x <= 1.  With w = x below 1/4 and w = 1/2 - x above (both exact), |w| <= 1/2,
// a = sin(pi w) = w P(w^2) and b = cos(pi w) = Q(w^2) (fit errors 2e-19 and 6e-21) are the two, in one order or the
// other (mean absolute error of (cs + 1) / 2: 2.5e-17, of a correctly rounded cosine 2.4e-17).  pi enters in two parts, its high part's product last, so that one rounding dominates.
__device__ __forceinline__ void sincospi_f64(double x, double& sn, double& cs) {
    const bool lo = x < 0.25;
    const double w = lo ? x : 0.5 - x, w2 = w * w;
    double p = 7.684026400701355e-07;
    p = fma_sc(p, w2, -2.190203105849926e-05);
    p = fma_sc(p, w2, 0.00046629917496286276);
    p = fma_sc(p, w2, -0.007370430357108927);
    p = fma_sc(p, w2, 0.08214588655343766);
    p = fma_sc(p, w2, -0.5992645293174708);
    p = fma_sc(p, w2, 2.550164039877242);
    p = fma_sc(p, w2, -5.1677127800499685);
    p = fma_sc(p, w2, 1.2246467991473532e-16);
    const double a = fma(w, 3.141592653589793, p * w);
    double q = -1.3435271577594177e-07;
    q = fma_sc(q, w2, 4.300724832508254e-06);
    q = fma_sc(q, w2, -0.0001046374171269161);
    q = fma_sc(q, w2, 0.0019295741873594852);
    q = fma_sc(q, w2, -0.0258068913766045);
    q = fma_sc(q, w2, 0.235330630357996);
    q = fma_sc(q, w2, -1.335262768854555);
    q = fma_sc(q, w2, 4.058712126416768);
    q = fma_sc(q, w2, -4.934802200544679);
    const double b = fma(q, w2, 1.0);
    sn = lo ? a : b;
    cs = lo ? b : a;
}

}  // namespace atomnn
