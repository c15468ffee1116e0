"""The reciprocals, roots and the viscosity law of hm_device.h, compiled for
the CPU with the hardware's estimates replaced by ones that are off by the
most that was measured of them, and without contraction of a*b + c: what the
source writes, the result may rest on, and nothing else.

Bounds (u = 2^-53): a reciprocal ends in one rounding, and its e + e^2 of 4.7e-8
adds 4.7e-8 u.  An inverse root's e = 1 - (d r) r carries the rounding of d r
(u, halved by the series) and ends in one: 1.5 u.  T^0.76 ends in the rounding
of 1 + q g (u for results over 1, u/2 of 0.707 below), after q g's own (u/4,
of 0.34) and g's (u/4 times ln 2): at most 1.7 u in all; 2 u = 2^-52 are
allowed."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
U = 2.0 ** -53

SHIM = r"""
#include <cmath>
#include <cstring>
#include <limits>
static double g_off = 0.0;  // relative error of the estimates
static double est_rcp(double d) { return 1.0 / d * (1.0 + g_off * 4.7e-8); }
static double est_rsq(double d) { return 1.0 / std::sqrt(d) * (1.0 + g_off * 5.5e-8); }
static double fix(double q, double d, double n) {  // special operands as a division has them
  if (d == 0.0 || std::isinf(d) || std::isnan(d)) return n / d;
  return std::copysign(std::fabs(q), std::signbit(d) != std::signbit(n) ? -1.0 : 1.0);
}
static long long as_ll(double x) { long long b; std::memcpy(&b, &x, 8); return b; }
static double as_d(long long b) { double x; std::memcpy(&x, &b, 8); return x; }
static int fexp(double x) { int e; std::frexp(x, &e); return e; }
static double fmant(double x) { int e; return std::frexp(x, &e); }
struct Dim { unsigned x; };
static Dim blockIdx, gridDim;
#define __device__
#define __host__
#define __forceinline__ inline
#define __builtin_amdgcn_rcp est_rcp
#define __builtin_amdgcn_rsq est_rsq
#define __builtin_amdgcn_div_fixup fix
#define __builtin_amdgcn_frexp_exp fexp
#define __builtin_amdgcn_frexp_mant fmant
#define __double_as_longlong as_ll
#define __longlong_as_double as_d
#define asm(...)
using std::fabs; using std::sqrt; using std::fmax;
#include "hm_device.h"
extern "C" {
void off(double x) { g_off = x; }
void rcp(const double *x, double *y, int n) { for (int i = 0; i < n; i++) y[i] = hm::nr_rcp(x[i]); }
void rsq(const double *x, double *y, int n) { for (int i = 0; i < n; i++) y[i] = hm::nr_rsq(x[i]); }
void root(const double *x, double *y, int n) { for (int i = 0; i < n; i++) y[i] = hm::nr_sqrt(x[i]); }
void pow76(const double *x, double *y, int n) { for (int i = 0; i < n; i++) y[i] = hm::pow076(x[i]); }
void prims(const double *u, double gamma, double *q) { hm::visc_prims(u, gamma, q); }
}
"""


@pytest.fixture(scope="module", params=[-1.0, 1.0])
def dev(request, tmp_path_factory):
    d = tmp_path_factory.mktemp("devmath")
    os.makedirs(d / "hip", exist_ok=True)
    (d / "hip" / "hip_runtime.h").write_text("")
    (d / "shim.cc").write_text(SHIM)
    so = d / "shim.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-shared", "-fPIC", "-I", str(d), "-I",
                    os.path.join(ROOT, "hypar_amd", "csrc"), str(d / "shim.cc"), "-o", str(so)], check=True)
    L = ctypes.CDLL(str(so))
    L.off.argtypes = [ctypes.c_double]
    L.off(request.param)
    L.prims.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_void_p]

    def call(name, x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        y = np.empty_like(x)
        getattr(L, name)(ctypes.c_void_p(x.ctypes.data), ctypes.c_void_p(y.ctypes.data), len(x))
        return y

    call.prims = lambda u, gamma: _prims(L, u, gamma)
    return call


def _prims(L, u, gamma):
    u = np.ascontiguousarray(u, dtype=np.float64)
    q = np.empty(4)
    L.prims(u.ctypes.data, gamma, q.ctypes.data)
    return q


def _arguments(lo, hi, n=200000):
    rng = np.random.default_rng(7)
    return np.exp2(rng.uniform(lo, hi, n))


def _error(got, exact):
    return float(np.abs((got.astype(np.longdouble) - exact) / exact).max())


def test_reciprocal_and_roots(dev):
    x = _arguments(-1000, 1000)
    X = x.astype(np.longdouble)
    assert _error(dev("rcp", x), 1 / X) <= 1.001 * U
    assert _error(dev("rsq", x), 1 / np.sqrt(X)) <= 1.51 * U
    assert _error(dev("root", x), np.sqrt(X)) <= 1.01 * U
    assert dev("root", np.zeros(1))[0] == 0.0


@pytest.mark.parametrize("lo,hi", [(-1, 1), (-44, 44), (-1022, 1023.99), (-1074, -1022)])
def test_viscosity_law(dev, lo, hi):
    x = _arguments(lo, hi)
    # both sides of the interval's ends sqrt(1/2) 2^k
    k = np.arange(int(np.ceil(lo)) + 1, int(hi))
    edge = np.sqrt(0.5) * np.exp2(k.astype(float))
    x = np.concatenate([x, edge, np.nextafter(edge, np.inf), np.nextafter(edge, 0), np.exp2(k.astype(float))])
    x = x[x > 0]
    exact = np.exp(np.longdouble(0.76) * np.log(x.astype(np.longdouble)))
    # the reference's own error: the logarithm's rounding, magnified by its size
    slack = 2.0 ** -64 * 0.76 * max(abs(lo), abs(hi)) + 2.0 ** -63
    assert _error(dev("pow76", x), exact) <= 2 * U + slack


def test_viscosity_law_special_values(dev):
    y = dev("pow76", [0.0, np.inf, np.nan, -1.0, -np.inf])
    assert y[0] == 0.0 and y[1] == np.inf and np.isnan(y[2:]).all()


@pytest.mark.parametrize("rho", [1.0, -2.0, 0.0, -0.0, np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("e", [2.5, 0.0, -1.0])
def test_viscous_primitives_divide(dev, rho, e):
    """u, v, w are zero without mass; beyond that the values are those of a division by rho."""
    gamma, m = 1.4, np.array([0.3, -0.2, 0.1])
    with np.errstate(all="ignore"):
        v = np.zeros(3) if rho == 0 else m / np.float64(rho)
        P = (e - 0.5 * np.float64(rho) * (v * v).sum()) * (gamma - 1)
        want = np.append(v, gamma * P / np.float64(rho))
    got = dev.prims([rho, *m, e], gamma)
    assert np.array_equal(np.isnan(got), np.isnan(want)), (got, want)
    ok = np.isfinite(want)
    assert np.array_equal(got[~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)])
    assert np.allclose(got[ok], want[ok], rtol=1e-14, atol=0)
