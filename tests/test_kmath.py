"""The scalar functions of the generated steps (hyx_kmath.hip): the roots of the step-size rule
and the half-integer powers, against extended precision, at the ends of their ranges."""

import ctypes as ct
import os
import subprocess

import numpy as np
import pytest

import heyoka_amd as hy
import pyoracle as O

CSRC = os.path.join(os.path.dirname(os.path.abspath(hy.__file__)), "csrc")
ROOTS = (1, 2, 11, 18, 19, 20, 200)
HARNESS = r"""
#include <cmath>
#include <math.h>
#define __device__
#define __forceinline__ inline
using std::sqrt; using std::pow;
#include "hyx_kmath.hip"
extern "C" {
""" + "".join(f"double root_{r}(double rn, double d) {{ return hyx_root<{r}>(rn, d); }}\n" for r in ROOTS) + r"""
double m32(double x, double *rx) { return hyx_pow_m3_2(x, *rx); }
double m12(double x, double *rx) { return hyx_pow_m1_2(x, *rx); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("kmath")
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "h.so"),
                    str(d / "h.cpp")], check=True, capture_output=True)
    return ct.CDLL(str(d / "h.so"))


def _args(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(lo, hi, n)


@pytest.mark.parametrize("r", ROOTS)
def test_root_against_extended_precision(lib, r):
    # q = den / num carries 2 roundings (half an ulp each), of which 1/r reach the root; the root's
    # own rounding, and that of y/r times the residual, add at most one ulp: 2^-52 (1 + 1/r).
    f = getattr(lib, f"root_{r}")
    f.restype, f.argtypes = ct.c_double, [ct.c_double] * 2
    den = _args(4000, -1000, 1000, r)
    num = np.where(np.arange(4000) % 3 == 0, 1.0, _args(4000, 0, 20, r + 1))
    got = np.array([f(1.0 / a, b) for a, b in zip(num, den)])
    ref = (num.astype(np.longdouble) / den) ** (np.longdouble(1) / r)
    ok = (ref < 1e308) & (ref > 1e-307)
    assert np.all(np.abs(got[ok] / ref[ok] - 1) <= 2.0 ** -52 * (1 + 1 / r))
    assert f(1.0, 0.0) == np.inf and f(1.0, np.inf) == 0.0 and np.isnan(f(1.0, np.nan)) and f(0.0, 3.0) == np.inf


@pytest.mark.parametrize("r", ROOTS)
def test_root_of_an_overflowing_quotient(lib, r):
    # num / den above the largest double: inf, as pow(num / den, 1 / r); just below it: finite.
    f = getattr(lib, f"root_{r}")
    f.restype, f.argtypes = ct.c_double, [ct.c_double] * 2
    for num, den in [(1.0, 1e-310), (1.0, 5e-324), (1e10, 1e-300), (1e200, 1e-200), (1.0, 2.0 ** -1024)]:
        with np.errstate(over="ignore"):
            assert np.float64(num) / den == np.inf
        assert f(1.0 / num, den) == np.inf, (num, den)
    for num, den in [(1.0, 2.0 ** -1023), (1.0, 2.0 ** -1022), (2.0 ** 500, 2.0 ** -522)]:
        ref = (np.longdouble(num) / den) ** (np.longdouble(1) / r)
        assert abs(f(1.0 / num, den) / ref - 1) <= 2.0 ** -52 * (1 + 1 / r), (num, den)


@pytest.mark.parametrize("name,al", [("m32", -1.5), ("m12", -0.5)])
def test_half_integer_powers(lib, name, al):
    f = getattr(lib, name)
    f.restype, f.argtypes = ct.c_double, [ct.c_double, ct.POINTER(ct.c_double)]
    rx = ct.c_double()
    edge = [2.0 ** -300, 2.0 ** 300, np.nextafter(2.0 ** -300, 1), np.nextafter(2.0 ** 300, 1), 1.0, 1e-200, 1e200]
    for x in list(_args(4000, -299, 299, 5)) + edge:
        y = f(x, ct.byref(rx))
        ref, rref = np.longdouble(x) ** np.longdouble(al), 1 / np.longdouble(x)
        assert abs(y / ref - 1) <= 2.0 ** -52 and abs(rx.value / rref - 1) <= 2.0 ** -52, x
    for x in (0.0, np.inf, -1.0, np.nan):
        with np.errstate(all="ignore"):
            ref = np.float64(x) ** al
        assert f(x, ct.byref(rx)) == ref or (np.isnan(ref) and np.isnan(f(x, ct.byref(rx)))), x


@pytest.mark.gpu
def test_half_integer_powers_on_the_device():
    x = hy.make_vars("x")
    cf = hy.cfunc([x ** -1.5, x ** -0.5, x ** -1.0], [x])
    v = np.concatenate([_args(5000, -1000, 1000, 7), [0.0, np.inf, -1.0, np.nan, 2.0 ** -300, 2.0 ** 300]])
    got = cf(v[None, :])
    with np.errstate(all="ignore"):
        ref = [v.astype(np.longdouble) ** np.longdouble(a) for a in (-1.5, -0.5, -1.0)]
        for g, r in zip(got, ref):
            r64 = r.astype(np.float64)
            fin = np.isfinite(r64) & (np.abs(r64) > 1e-300)
            assert np.all(np.abs(g[fin] / r[fin] - 1) <= 2.0 ** -52)
            rest = ~fin & (np.abs(r64) > 1e-300)
            assert np.array_equal(g[rest], r64[rest]) and np.array_equal(np.isnan(g), np.isnan(r64))


@pytest.mark.gpu
@pytest.mark.parametrize("amp", [0.0, 1e-300, 1e-100, 1.0, 1e100, 1e300, np.inf, np.nan])
def test_step_size_over_the_exponent_range(amp):
    # The oracle's h comes from pow(num / mo, 1 / p), whose exponent is rounded: an error of up
    # to |log(num / mo)| 2^-53 / p, at most 690 * 2^-53 / 19, beside its own and the norms' rounding.
    xs, v = hy.make_vars("x", "v")
    sys_ = [(xs, v), (v, -xs)]
    st = np.array([[amp], [0.5 * amp]])
    ta = hy.taylor_adaptive_batch(sys_, st, tol=1e-15)
    ta.step(np.array([1e3]))
    r = O.step_batch(hy.taylor_decompose(sys_), 19, st, max_dt=np.array([1e3]))
    assert int(ta.step_res[0][0]) == int(r["outcome"][0])
    assert abs(ta.last_h[0] - r["h"][0]) <= 1e-14 * abs(r["h"][0])


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["unrolled", "compact", "group", "wave"])
@pytest.mark.parametrize("amp", [1e-300, 1e-290, 1e-280])
def test_free_step_of_a_tiny_state(amp, form):
    # Without a step limit: order 19 of a state of 1e-300 is 1e-317, whose quotient overflows (the step
    # is infinite and its state not finite, as in the oracle); from 1e-290 on it does not.
    x, y, vx, vy = hy.make_vars("x", "y", "vx", "vy")
    sys_ = [(x, vx), (y, vy), (vx, -x * 1.5), (vy, -y * 1.5)]
    if form == "group":
        sys_ = [(x, vx), (y, vy), (vx, hy.sin(x) * -1.5), (vy, hy.sin(y) * -1.5)]
    st = np.array([[amp], [0.5 * amp], [amp], [0.5 * amp]])
    ta = hy.taylor_adaptive_batch(sys_, st, tol=1e-15, code_form=form)
    ta.step()
    r = O.step_batch(hy.taylor_decompose(sys_), 19, st)
    assert int(ta.step_res[0][0]) == int(r["outcome"][0])
    if np.isfinite(r["h"][0]):
        assert abs(ta.last_h[0] - r["h"][0]) <= 1e-13 * abs(r["h"][0])
    else:
        assert ta.last_h[0] == r["h"][0]
