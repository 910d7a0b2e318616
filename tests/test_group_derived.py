"""The group form where the cluster inputs are derived variables (x' = v): positions stored at
order 0 only, masses folded into the owners' sums, two waves per SIMD. Body counts whose
pairs fill a group or leave lanes over, orders on both sides of the two-wave rule, and
systems that keep the general layout (an input that is not a lone derivative)."""

import ctypes as ct
import subprocess

import numpy as np
import pytest

import heyoka_amd as hy
import pyoracle as O
from heyoka_amd import _lib
from test_codegen_cpu import GROUP_HARNESS


def _nbody(n, massless=0):
    rng = np.random.default_rng(n)
    m = [1.0] + list(rng.uniform(1e-3, 0.2, n - 1))
    for i in range(massless):
        m[n - 1 - i] = 0.0
    st = np.zeros(6 * n)
    for i in range(n):
        th = 2.4 * i
        r = 1.5 * i
        st[6 * i:6 * i + 3] = [r * np.cos(th), r * np.sin(th), 0.1 * (i % 3)]
        if i:
            st[6 * i + 3:6 * i + 5] = np.array([-np.sin(th), np.cos(th)]) / np.sqrt(r)
    return hy.model.nbody(n, masses=m), st


def _drag(n=3):
    # Isomorphic clusters over pairs whose inputs include the velocities.
    xs, vs = hy.make_vars(*[f"x{i}" for i in range(n)]), hy.make_vars(*[f"v{i}" for i in range(n)])
    acc = [[] for _ in range(n)]
    for i in range(n):
        for j in range(i + 1, n):
            f = (vs[j] - vs[i]) * ((xs[j] - xs[i]) ** 2 + 1.0) ** -1.5
            acc[i].append(0.5 * f)
            acc[j].append(-0.25 * f)
    sys_ = [(x, v) for x, v in zip(xs, vs)] + [(v, acc[i][0] + acc[i][1]) for i, v in enumerate(vs)]
    return sys_, np.concatenate([np.arange(n) * 0.7, 0.3 - 0.4 * np.arange(n) ** 2])


CASES = {"n3": lambda: _nbody(3), "n4": lambda: _nbody(4), "n5": lambda: _nbody(5), "n6": lambda: _nbody(6),
         "n8": lambda: _nbody(8), "drag": lambda: _drag()}


@pytest.mark.parametrize("p", [5, 12, 20, 24])
@pytest.mark.parametrize("name", list(CASES))
def test_group_step_cpu(name, p, tmp_path):
    sys_, st = CASES[name]()
    dec = hy.taylor_decompose(sys_)
    src = _lib.System(dec, p, compact="group", source_only=True).source()
    if name == "n6":
        assert ("#define HYX_GROUP_WAVES 2" in src) == (p <= 20)
    if name == "drag":  # its clusters read velocities: no derived variables, slots as variables
        assert "#define HYX_OWN 2\n" in src and "#define HYX_NX 7\n" in src
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
@pytest.mark.parametrize("tol", [1e-9, 1e-15, 0.0])
@pytest.mark.parametrize("name", list(CASES))
def test_group_propagation(name, tol):
    sys_, st0 = CASES[name]()
    N = 37
    st = np.repeat(st0[:, None], N, axis=1) + np.random.default_rng(1).normal(0.0, 1e-3, (len(st0), N))
    print(f"[gpu] group {name} tol={tol}", flush=True)
    out = {}
    for mode in ("persistent", "plain"):
        ta = hy.taylor_adaptive_batch(sys_, st, tol=tol, code_form="group", gpu_mode=mode)
        ta.propagate_until(np.linspace(0.5, 2.0, N))
        out[mode] = (ta.state.copy(), ta.propagate_res)
    assert np.array_equal(out["persistent"][0], out["plain"][0]) and out["persistent"][1] == out["plain"][1]
    r = O.propagate_until(hy.taylor_decompose(sys_), ta.order, st, np.linspace(0.5, 2.0, N))
    np.testing.assert_allclose(out["plain"][0], r["state"], rtol=1e-10, atol=1e-10)
    assert [x[3] for x in out["plain"][1]] == list(r["nsteps"])
