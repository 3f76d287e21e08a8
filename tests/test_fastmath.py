"""The FP64 exponential, tanh and cutoff sine and cosine of the kernels (atomnn_amd/csrc/fastmath.hpp), built for the
host (the same steps; the hardware's approximate reciprocal in tanh stands as a float's) and compared with 80-bit long
double on 3 million points a range, its ends, halves and quarters among them.  The bounds follow from the forms: each has a
last rounding of 0.5 ulp, and before it
  e^x          two roundings of r (ulp(r) / 2 <= 2^-55 each, 0.25 ulp of a result below 1) and the one of 1 + r q, times |r| <= 0.35:
               0.5 + 2 * 0.25 + 0.35 = 1.35 ulp at worst; subnormal results are rounded twice
  sin, cos     the rounding of w^2 and of the polynomial, times 4.7 w^2 <= 0.3: below 0.6 ulp more, 1.1 in all
  tanh z       m to 1.35 ulp of e^r - 1, halved or less by d t / d m = 2 / (2 + m)^2 <= 1 near 0, the sum 2 + m and the quotient
               0.5 each, and a change of binade that doubles the ulp: 3 ulp, as the kernels' users are told."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cmath>
#include "fastmath.hpp"
using namespace atomnn;
extern "C" double value(int f, double x) {
    double s, c;
    if (f == 0) return exp_f64(x);
    if (f == 1) return tanh_f64(x);
    sincospi_f64(x, s, c);
    return f == 2 ? s : c;
}
static long double exact(int f, double x) {
    const long double v = x;
    if (f == 0) return expl(v);
    if (f == 1) return tanhl(v);
    const long double pi = 3.14159265358979323846264338327950288L;
    if (f == 2) return sinl(pi * (v > 0.5L ? 1 - v : v));
    return v < 0.25L ? cosl(pi * v) : v > 0.75L ? -cosl(pi * (1 - v)) : sinl(pi * (0.5L - v));
}
// largest and rms error in ulp of the exact value, largest absolute error
extern "C" void errors(int f, const double* x, long n, double* out) {
    double mx = 0, sq = 0, ab = 0;
    for (long i = 0; i < n; ++i) {
        const long double t = exact(f, x[i]);
        const double e = (double)fabsl((long double)value(f, x[i]) - t), a = (double)fabsl(t);
        const double u = e / (std::nextafter(a, INFINITY) - a);
        if (!(u <= mx)) mx = u;  // (a NaN shows)
        if (!(e <= ab)) ab = e;
        sq += u * u;
    }
    out[0] = mx;
    out[1] = std::sqrt(sq / n);
    out[2] = ab;
}
"""


@pytest.fixture(scope="module")
def fm(tmp_path_factory):
    d = tmp_path_factory.mktemp("fastmath")
    src, so = str(d / "fm.cpp"), str(d / "fm.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "atomnn_amd", "csrc"), "-o", so, src], check=True)
    lib = ctypes.CDLL(so)
    lib.value.argtypes, lib.value.restype = [ctypes.c_int, ctypes.c_double], ctypes.c_double
    lib.errors.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_long, ctypes.c_void_p]
    return lib


def errors(fm, f, lo, hi, also=()):
    rng = np.random.default_rng(f)
    x = np.concatenate([rng.uniform(lo, hi, 3_000_000), [lo, hi], np.linspace(lo, hi, 4097), also])
    out = np.zeros(3)
    fm.errors(f, x.ctypes.data, len(x), out.ctypes.data)
    return out


EXP, TANH, SIN, COS = range(4)


@pytest.mark.parametrize("lo,hi", [(-0.35, 0.35), (-1.0, 0.0), (-100.0, 0.0), (-708.0, -100.0), (0.0, 709.0)])
def test_exponential(fm, lo, hi):
    mx, rms, _ = errors(fm, EXP, lo, hi)
    assert mx <= 1.35 and rms <= 0.32  # a correctly rounded result has 0.289 rms


def test_exponential_beyond_the_normal_range(fm):
    assert errors(fm, EXP, -745.0, -708.5)[0] <= 2.0
    for x in (-750.0, -1000.0, -1e6, -1e300, -np.inf):
        assert fm.value(EXP, x) == 0.0
    assert fm.value(EXP, 0.0) == 1.0 and fm.value(EXP, -0.0) == 1.0
    assert fm.value(EXP, 710.0) == np.inf and np.isnan(fm.value(EXP, np.nan))


@pytest.mark.parametrize("lo,hi", [(-1e-300, 1e-300), (-1e-6, 1e-6), (-0.18, 0.18), (-1.0, 1.0), (-22.0, 22.0)])
def test_tanh(fm, lo, hi):
    assert errors(fm, TANH, lo, hi)[0] <= 3.0


def test_tanh_limits(fm):
    for x in (25.0, 400.0, 1e6, 1e300, np.inf):
        assert fm.value(TANH, x) == 1.0 and fm.value(TANH, -x) == -1.0
    assert fm.value(TANH, 0.0) == 0.0 and np.signbit(fm.value(TANH, -0.0)) and np.isnan(fm.value(TANH, np.nan))


@pytest.mark.parametrize("f", [SIN, COS])
@pytest.mark.parametrize("lo,hi", [(1e-12, 1.0 - 2.0**-53), (1e-12, 0.001), (0.2499, 0.2501), (0.4999, 0.49999999),
                                   (0.50000001, 0.5001), (0.7499, 0.7501), (0.999, 1.0 - 2.0**-53)])
def test_cutoff_sine_and_cosine(fm, f, lo, hi):
    mx, rms, ab = errors(fm, f, lo, hi)
    assert mx <= 1.1 and ab <= 1.1 * 2.0**-53
    if hi - lo > 0.9:
        assert rms <= 0.31


def test_sine_and_cosine_at_the_quarters(fm):
    for x, s, c in ((0.0, 0.0, 1.0), (0.5, 1.0, 0.0), (1.0, 0.0, -1.0)):
        assert fm.value(SIN, x) == s and fm.value(COS, x) == c
    e = 2.0**-52  # a distance a last place beyond the cutoff
    assert abs(fm.value(SIN, 1.0 + e) + np.pi * e) <= 1e-30 and fm.value(COS, 1.0 + e) == -1.0
