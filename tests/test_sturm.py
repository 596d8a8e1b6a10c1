"""The extreme eigenvalue of a Lanczos tridiagonal (csrc/sq_sturm.hpp), compiled for
the CPU, against bisection in long double: no less accurate than the same iteration
with divisions, run until no step moves inward."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sqdft_amd", "csrc")

SRC = r"""
#include "sq_sturm.hpp"
#include <algorithm>
#include <cmath>
extern "C" {
// 1/q as the kernel forms it: an estimate (here the division with its last 29 bits
// cut off) and two Newton steps
static double recip(double q)
{
    union { double d; unsigned long u; } v{1.0 / q};
    v.u &= ~0x1ffffffful;
    double r = v.d;
    r = std::fma(std::fma(-q, r, 1.0), r, r);
    return std::fma(std::fma(-q, r, 1.0), r, r);
}
int largest(const double *d, const double *e, int n, double sg, double f, double b, double g, double *out)
{
    return sqk::tridiag_largest([&](int i) { return d[i]; }, [&](int i) { return e[i]; }, recip, n, sg, f, b, g, out);
}
double divided(const double *d, const double *e, int n, double sg, double x)
{
    for (;;) {
        double q = x - sg * d[0], dq = 1.0, iq = 1.0 / q, s = iq;
        for (int i = 1; i < n; ++i) {
            const double r = e[i - 1] * e[i - 1] * iq;
            dq = 1.0 + r * dq * iq;
            q = (x - sg * d[i]) - r;
            iq = 1.0 / q;
            s += dq * iq;
        }
        const double xn = x - 1.0 / s;
        if (!(xn < x)) return x;
        x = xn;
    }
}
// error of x as the largest eigenvalue, by bisection from f (outside)
double error(const double *d, const double *e, int n, double sg, double f, double x)
{
    long double hi = f, lo = sg * d[0];
    for (int i = 1; i < n; ++i) lo = std::max(lo, (long double)(sg * d[i]));
    lo -= 1e-9L;
    for (int it = 0; it < 120; ++it) {
        const long double m = (lo + hi) / 2;
        long double q = m - (long double)(sg * d[0]);
        bool out = q > 0;
        for (int i = 1; i < n && out; ++i) {
            q = (m - (long double)(sg * d[i])) - (long double)e[i - 1] * e[i - 1] / q;
            out = q > 0;
        }
        (out ? hi : lo) = m;
    }
    return (double)fabsl((long double)x - hi);
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("sturm")
    src = d / "sturm.cpp"
    src.write_text(SRC)
    so = d / "libsturm.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC,
                    str(src), "-o", str(so)], check=True)
    L = C.CDLL(str(so))
    P, D, I = C.POINTER(C.c_double), C.c_double, C.c_int
    L.largest.argtypes = [P, P, I, D, D, D, D, P]
    L.divided.argtypes = [P, P, I, D, D]
    L.divided.restype = D
    L.error.argtypes = [P, P, I, D, D, D]
    L.error.restype = D
    return L


def _ptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


@pytest.mark.parametrize("far", [True, False])
@pytest.mark.parametrize("centre", [0.0, 0.5, 40.0])
def test_extremes_as_accurate_as_with_divisions(lib, centre, far):
    rng = np.random.default_rng(7)
    new, old = [], []
    for _ in range(600):
        n = int(rng.integers(2, 120))
        w = float(rng.uniform(1.0, 20.0))
        d = centre + 0.3 * w * rng.uniform(-1, 1, n) * np.exp(-0.05 * np.arange(n))
        e = w * rng.uniform(0.25, 0.45, n - 1)
        rad = np.concatenate([[0.0], e]) + np.concatenate([e, [0.0]])
        size = abs(centre) + w
        for sg in (1.0, -1.0):
            f = float(np.max(sg * d + rad)) + 1e-14 * size
            near = lib.divided(_ptr(d), _ptr(e), n, sg, f)
            x = C.c_double()
            b, g = (f, 1.0) if far else (near - 1e-7 * size, 1e-9 * size)   # the near start begins inside
            assert lib.largest(_ptr(d), _ptr(e), n, sg, f, b, g, C.byref(x))
            new.append(lib.error(_ptr(d), _ptr(e), n, sg, f, x.value) / size)
            old.append(lib.error(_ptr(d), _ptr(e), n, sg, f, near) / size)
    rms = [float(np.sqrt(np.mean(np.square(v)))) for v in (new, old)]
    # the same error up to the scatter of 1,200 last-bit roundings (a few per cent);
    # a stop that leaves out the last step has a quarter to a half more
    assert rms[0] <= 1.1 * rms[1], rms
    assert max(new) <= 2.3e-16
