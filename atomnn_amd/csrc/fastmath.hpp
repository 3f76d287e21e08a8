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
__host__ __device__ __forceinline__ double fma_sc(double a, double b, double c) {
#ifdef __HIP_DEVICE_COMPILE__
    double o;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(o) : "v"(a), "v"(b), "s"(c));
    return o;
#else
    return fma(a, b, c);
#endif
}

// An approximate 1 / d, about as good as a float (v_rcp_f64).
__host__ __device__ __forceinline__ double rcp_approx(double d) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcp(d);
#else
    return (double)(float)(1.0 / d);
#endif
}

// e^x.  x = n ln 2 + r, |r| <= ln 2 / 2; e^r = 1 + r (1 + r q(r)), q of degree 9 (fit error 3.6e-18); below -1000
// (where e^x is 0 in FP64) the argument is held, so that infinite products give 0.  On 4 million points
// of [-100, 0] the error is 0.91 ulp at most and 0.302 ulp rms (the library's 0.87 and 0.302), of [-1, 0] 0.81 and 0.300
// (0.84 and 0.301).
__host__ __device__ __forceinline__ double exp_f64(double x) {
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
// instructions (expm1 and the compiler's division: about 90), and the same errors, up to 2.5 ulp.
__host__ __device__ __forceinline__ double tanh_f64(double z) {
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
    double y = rcp_approx(d);
    y = fma(fma(-d, y, 1.0), y, y);
    y = fma(fma(-d, y, 1.0), y, y);
    double t = -m * y;
    t = fma(fma(-d, t, -m), y, t);
    return copysign(t, z);
}

// sin(pi x) and cos(pi x) for 0 <= x <= 1 (a last place beyond is fine).  With n = 0, 1 or 2 the integer nearest 2 x and
// w = x - n / 2 (exact), |w| <= 1/4, a = sin(pi w) = w P(w^2) and b = cos(pi w) = 1 + w^2 Q(w^2) (fit errors 2e-18 and
// 4e-20) are the two up to order and sign.  pi enters in two parts, its high part's product last, so that one rounding
// dominates.  On 4 million points the errors are 1.0 ulp at most and 0.301 ulp rms (the library's 0.88 and 0.301).  Two
// polynomials over |w| <= 1/2 instead cancel near the cutoff: 2.1 ulp of the cosine, 2.4e-16 of the sine near its zero.
__host__ __device__ __forceinline__ void sincospi_f64(double x, double& sn, double& cs) {
    const double n = rint(x + x), w = fma(-0.5, n, x), w2 = w * w;
    double p = 0.00046119481320414514;
    p = fma_sc(p, w2, -0.007369953143376355);
    p = fma_sc(p, w2, 0.08214586383478734);
    p = fma_sc(p, w2, -0.5992645287393041);
    p = fma_sc(p, w2, 2.550164039869727);
    p = fma_sc(p, w2, -5.167712780049926);
    p = fma_sc(p, w2, 4.92452851378537e-17);
    const double a = fma(w, 3.141592653589793, p * w);
    double q = -0.00010357918388694153;
    q = fma_sc(q, w2, 0.0019294684683380183);
    q = fma_sc(q, w2, -0.02580688590585543);
    q = fma_sc(q, w2, 0.235330630202802);
    q = fma_sc(q, w2, -1.3352627688522163);
    q = fma_sc(q, w2, 4.058712126416751);
    q = fma_sc(q, w2, -4.934802200544679);
    const double b = fma(q, w2, 1.0);
    const double s = n == 1.0 ? b : a, c = n == 1.0 ? a : b;
    sn = n > 1.0 ? -s : s;
    cs = n > 0.0 ? -c : c;
}

}  // namespace atomnn
