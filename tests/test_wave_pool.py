"""The wave form's pool (sums over lower orders spread over all lanes) and its derived state
variables: systems whose sums fill less than one pool slot, exactly one, several; with and
without variables that follow from another's right-hand side; orders from the lowest to
beyond 20; every lane count. One step on the CPU emulation against the oracle."""

import ctypes as ct
import subprocess

import numpy as np
import pytest

import heyoka_amd as hy
import pyoracle as O
from heyoka_amd import _lib
from test_codegen_cpu import GROUP_HARNESS


def _products(n, second):
    """n coupled variables with a product, a square or a power each; second: as accelerations."""
    xs = hy.make_vars(*[f"x{i}" for i in range(n)])
    vs = hy.make_vars(*[f"v{i}" for i in range(n)])
    f = []
    for i in range(n):
        a, b = xs[i], xs[(i + 1) % n]
        f.append([0.3 * (a * b), -0.2 * (a ** 2) * b, (a * a + 1.5) ** -1.5 * b, (b * b + 1.2) ** -0.5 - 0.1 * a][i % 4])
    x0 = 0.4 + 0.3 * np.cos(np.arange(n))
    if not second:
        return list(zip(xs, f)), x0
    return list(zip(xs, vs)) + list(zip(vs, f)), np.concatenate([x0, 0.1 * np.sin(np.arange(n))])


CASES = {"1st_3": (3, False), "1st_16": (16, False), "2nd_4": (4, True), "2nd_17": (17, True), "2nd_33": (33, True)}


@pytest.mark.parametrize("form", ["wave", "wave32", "wave16"])
@pytest.mark.parametrize("p", [2, 3, 4, 5, 12, 24])
@pytest.mark.parametrize("name", list(CASES))
def test_wave_pool_step(name, p, form, tmp_path):
    sys_, st = _products(*CASES[name])
    dec = hy.taylor_decompose(sys_)
    src = _lib.System(dec, p, compact=form, source_only=True).source()
    (tmp_path / "prelude.inc").write_text(src.split("// Hand-written CDNA4 kernels")[0])
    (tmp_path / "g.cpp").write_text(GROUP_HARNESS)
    so = tmp_path / "g.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-pthread", "-o", str(so),
                    str(tmp_path / "g.cpp")], check=True, capture_output=True)
    L = ct.CDLL(str(so))
    P = ct.POINTER(ct.c_double)
    L.gstep_cpu.argtypes = [P, P, ct.c_double, ct.c_double, P, P, ct.POINTER(ct.c_int), P]
    n = dec.n_state
    xout, h, nf, tc, pv = np.zeros(n), np.zeros(64), np.zeros(64, dtype=np.int32), np.zeros(n * (p + 1)), np.zeros(1)
    ptr = lambda a: a.ctypes.data_as(P)  # noqa: E731
    G = L.gstep_cpu(ptr(st), ptr(pv), 0.0, np.inf, ptr(xout), ptr(h), nf.ctypes.data_as(ct.POINTER(ct.c_int)), ptr(tc))
    assert np.all(h[:G] == h[0]) and not nf[:G].any()
    r = O.step_batch(dec, p, st[:, None], want_tc=True)
    tco = r["tc"][:, :, 0]
    scale = np.max(np.abs(tco), axis=1, keepdims=True) + 1e-300
    assert np.max(np.abs(tc.reshape(n, p + 1) - tco) / scale) < 1e-11
    assert abs(h[0] - r["h"][0]) <= 1e-13 * abs(r["h"][0])
    np.testing.assert_allclose(xout, r["state"][:, 0], rtol=1e-13, atol=1e-15)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_wave_pool_propagation(name):
    sys_, st0 = _products(*CASES[name])
    N = 29
    st = np.repeat(st0[:, None], N, axis=1) + np.random.default_rng(3).normal(0.0, 1e-2, (len(st0), N))
    tf = np.linspace(0.3, 1.5, N)
    print(f"[gpu] wave pool {name}", flush=True)
    out = []
    for form in ("wave", "wave32", "wave16"):
        ta = hy.taylor_adaptive_batch(sys_, st, tol=1e-15, code_form=form)
        grid = np.linspace(0.0, 1.0, 5)[:, None] * tf
        _, g = ta.propagate_grid(grid)
        out.append((ta.state.copy(), g))
    # The lane counts compute every node alike.
    assert all(np.array_equal(a, out[0][0]) and np.array_equal(b, out[0][1]) for a, b in out[1:])
    r = O.propagate_grid(hy.taylor_decompose(sys_), 19, st, grid)
    np.testing.assert_allclose(out[0][1], r["out"], rtol=1e-11, atol=1e-12)
