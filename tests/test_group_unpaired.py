"""The group form with state variables that have no derived one (x' = v) beside others that do:
their lanes leave a derived slot empty, which must read +0.0 over the steps of a propagation (the
persistent kernel keeps it in registers) and must not enter the norms of the step-size rule."""

import ctypes as ct
import subprocess

import numpy as np
import pytest

import heyoka_amd as hy
import pyoracle as O
from heyoka_amd import _lib
from test_codegen_cpu import GROUP_HARNESS

# Steps in sequence, the owned variables (and what the empty slots hold) kept from one to the next.
MULTI = GROUP_HARNESS + r"""
struct MArg { int g; const double *x; const double *pv; int ns; double *xout; double *h; };
static void *mrun(void *p)
{
    MArg *a = (MArg *)p;
    tl_g = a->g;
    hyx_gtab t;
    hyx_gtab_load(t, a->g);
    double xo[HYX_OWN], pv[HYX_NPAR] = {};
    for (int o = 0; o < HYX_OWN; ++o) xo[o] = (t.vo[o] >= 0) ? a->x[t.vo[o]] : 0.0;
    for (int s = 0; s < a->ns; ++s) {
        double h; bool nf;
        hyx_gstep<false>(xo, pv, 0.0, INFINITY, h, nf, a->g, fl, t, nullptr, 1);
        for (int o = 0; o < HYX_OWN; ++o) if (t.vo[o] >= 0) a->xout[s * HYX_N + t.vo[o]] = xo[o];
        if (a->g == 0) a->h[s] = h;
    }
    return nullptr;
}
extern "C" void gsteps_cpu(const double *x, const double *pv, int ns, double *xout, double *h)
{
    for (int q = 0; q < HYX_FLAT; ++q) fl[q] = 0.0;
    pthread_barrier_init(&bar, nullptr, HYX_G);
    pthread_t th[HYX_G]; MArg args[HYX_G];
    for (int g = 0; g < HYX_G; ++g) { args[g] = MArg{g, x, pv, ns, xout, h}; pthread_create(&th[g], nullptr, mrun, &args[g]); }
    for (int g = 0; g < HYX_G; ++g) pthread_join(th[g], nullptr);
    pthread_barrier_destroy(&bar);
}
"""


def _system(bodies, extra, unit):
    """N bodies with the time unit scaled by `unit`, and extra equations: `w` the integral of a
    velocity, `const` a linear function of time, `chain` a variable whose derivative is w, `quad`
    one variable per velocity integrating its acceleration again (every lane of a slot)."""
    rng = np.random.default_rng(bodies)
    m = np.array([1.0] + list(rng.uniform(1e-3, 0.2, bodies - 1))) / unit ** 2
    sys_ = list(hy.model.nbody(bodies, masses=list(m)))
    st = np.zeros(6 * bodies)
    for i in range(bodies):
        th, r = 2.4 * i, 1.5 * i
        st[6 * i:6 * i + 3] = [r * np.cos(th), r * np.sin(th), 0.1 * (i % 3)]
        if i:
            st[6 * i + 3:6 * i + 5] = np.array([-np.sin(th), np.cos(th)]) / np.sqrt(r) / unit
    names = [str(v) for v, _ in sys_]
    vx1, dvx0 = sys_[names.index("vx_1")][0], sys_[names.index("vx_0")][1]
    w, c, w2 = hy.make_vars("w", "c", "w2")
    more, x0 = [], []
    if "w" in extra:
        more.append((w, vx1))
        x0.append(0.3)
    if "const" in extra:
        more.append((c, hy.expression(0.5 / unit)))
        x0.append(-0.2)
    if "chain" in extra:
        more.append((w2, w))
        x0.append(0.1)
    if "quad" in extra:
        more += list(zip(hy.make_vars(*[f"q{i}" for i in range(3)]),
                         [dvx0, sys_[names.index("vy_0")][1], sys_[names.index("vx_1")][1]]))
        x0 += [0.01 / unit, 0.02 / unit, -0.01 / unit]
    return sys_ + more, np.concatenate([st, x0])


EXTRAS = [("w",), ("const",), ("w", "chain"), ("w", "const", "chain"), ("quad",), ("w", "quad")]


@pytest.mark.parametrize("unit", [1.0, 1000.0])
@pytest.mark.parametrize("ha", [False, True])
@pytest.mark.parametrize("bodies,extra", [(3, e) for e in EXTRAS] + [(4, ("w", "const")), (5, ("w",)),
                                          (6, ("w", "const", "chain")), (7, ("w", "quad"))])
def test_steps_in_sequence_match_the_oracle(bodies, extra, ha, unit, tmp_path):
    sys_, st = _system(bodies, extra, unit)
    dec, p, ns = hy.taylor_decompose(sys_), 20, 5
    s = _lib.System(dec, p, high_accuracy=ha, compact="group", source_only=True)
    assert s.form == "group"
    (tmp_path / "prelude.inc").write_text(s.source().split("// Hand-written CDNA4 kernels")[0])
    (tmp_path / "g.cpp").write_text(MULTI)
    so = tmp_path / "g.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-pthread", "-o", str(so),
                    str(tmp_path / "g.cpp")], check=True, capture_output=True)
    L = ct.CDLL(str(so))
    n = dec.n_state
    xout, h, pv = np.zeros((ns, n)), np.zeros(ns), np.zeros(1)
    ptr = lambda a: a.ctypes.data_as(ct.POINTER(ct.c_double))  # noqa: E731
    L.gsteps_cpu(ptr(st), ptr(pv), ns, ptr(xout), ptr(h))
    x = st[:, None]
    for q in range(ns):
        # A step's rounding is some units of 2^-53 per variable, and the five steps (a fraction of a
        # period) enlarge a difference by less than ten; h is a 19th root of order p's norm, whose
        # terms cancel by up to 1e4 in the worst body pair.
        r = O.step_batch(dec, p, x, high_accuracy=ha)
        x = r["state"]
        assert abs(h[q] - r["h"][0]) <= 1e-11 * abs(r["h"][0]), (q, h[q], r["h"][0])
        scale = np.maximum(np.abs(x[:, 0]), 1.0 / unit)
        assert np.max(np.abs(xout[q] - x[:, 0]) / scale) < 1e-12, q


@pytest.mark.gpu
@pytest.mark.parametrize("ha", [False, True])
@pytest.mark.parametrize("bodies,extra", [(3, ("w", "quad")), (5, ("w",)), (6, ("w", "const", "chain"))])
def test_propagation_keeps_the_state(bodies, extra, ha):
    sys_, st0 = _system(bodies, extra, 1.0)
    N = 37
    st = np.repeat(st0[:, None], N, axis=1) + np.random.default_rng(1).normal(0.0, 1e-3, (len(st0), N))
    tf = np.linspace(0.5, 2.0, N)
    print(f"[gpu] group unpaired bodies={bodies} {extra} ha={ha}", flush=True)
    out = {}
    for mode in ("persistent", "plain"):
        ta = hy.taylor_adaptive_batch(sys_, st, tol=1e-15, high_accuracy=ha, code_form="group", gpu_mode=mode)
        ta.propagate_until(tf)
        out[mode] = (ta.state.copy(), ta.propagate_res)
    assert np.array_equal(out["persistent"][0], out["plain"][0]) and out["persistent"][1] == out["plain"][1]
    r = O.propagate_until(hy.taylor_decompose(sys_), ta.order, st, tf, high_accuracy=ha)
    np.testing.assert_allclose(out["plain"][0], r["state"], rtol=1e-10, atol=1e-10)
    assert [x[3] for x in out["plain"][1]] == list(r["nsteps"])
