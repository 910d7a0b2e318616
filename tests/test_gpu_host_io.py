"""State, parameters, times and results of a batch in one call: through the pinned image of small
batches and through the caller's arrays of larger ones, against the calls per field."""

import numpy as np
import pytest

import heyoka_amd as hy
from heyoka_amd import _lib, workloads
from test_zz_no_alloc import D2H, _hip

pytestmark = pytest.mark.gpu


def _system(name):
    if name == "cr3bp":  # one runtime parameter
        return hy.model.cr3bp_planar(), 4, 1
    return hy.model.pendulum(), 2, 0


# The image (used from the second time on that a batch is filled) holds 15 doubles per instance of
# the CR3BP and 12 of the pendulum, up to 256 KB: 2,100 and 2,800 lie on either side for both.
@pytest.mark.parametrize("name", ["cr3bp", "pendulum"])
@pytest.mark.parametrize("n", [1, 31, 33, 2100, 2800])
def test_all_fields_at_once(name, n):
    eqs, dim, npar = _system(name)
    rng = np.random.default_rng(n)
    st = rng.uniform(-0.1, 0.1, (dim, n)) + np.array([[0.48], [0.85], [0.0], [0.0]])[:dim]
    pa = rng.uniform(0.004, 0.012, (npar, n))
    thi, tlo = rng.uniform(-1.0, 1.0, n), rng.uniform(-1e-17, 1e-17, n)
    s = _lib.System(hy.taylor_decompose(eqs), 20)
    one, other = _lib.Batch(s, n), _lib.Batch(s, n)
    for rep in range(3):
        st = st + 0.001 * rep
        one.write_all(st, pa, thi, tlo)
        one.write_all(st, pa, thi, tlo)  # nothing waited for in between
        other.write(_lib.FIELD_STATE, st)
        if npar:
            other.write(_lib.FIELD_PARS, pa)
            assert np.array_equal(one.read(_lib.FIELD_PARS, pa.shape), pa)
        other.write(_lib.FIELD_TIME_HI, thi)
        other.write(_lib.FIELD_TIME_LO, tlo)
        for f, v in ((_lib.FIELD_STATE, st), (_lib.FIELD_TIME_HI, thi), (_lib.FIELD_TIME_LO, tlo)):
            assert np.array_equal(one.read(f, v.shape), v)
        tf = thi + rng.uniform(0.5, 3.0, n)
        lim = None if rep == 0 else np.full(n, 0.2 * rep)
        one.propagate_until(tf, None, lim, want_res=False)
        want = other.propagate_until(tf, None, lim)
        got = np.empty((dim, n)), np.empty(n), np.empty(n)
        res = np.empty(n, np.int64), np.empty(n), np.empty(n), np.empty(n, np.uint64)
        one.read_all(*got, res)
        for f, v in zip((_lib.FIELD_STATE, _lib.FIELD_TIME_HI, _lib.FIELD_TIME_LO), got):
            assert np.array_equal(other.read(f, v.shape), v)
        for k, v in zip(("outcome", "min_h", "max_h", "nsteps"), res):
            assert np.array_equal(want[k], v)
        # Without results, into an array that is not contiguous.
        wide = np.zeros((dim, n + 1))
        one.read_all(wide[:, :n], *got[1:])
        assert np.array_equal(wide[:, :n], got[0]) and not wide[:, n].any()


@pytest.mark.parametrize("row, col, msg", [(3, 4, "non-monotonic"), (1, 0, "non-monotonic"), (0, 2, "does not match")])
def test_grid_faults_name_the_instance(row, col, msg):
    wl = workloads.cr3bp(7)
    s = _lib.System(hy.taylor_decompose(wl.sys), 18)
    b = _lib.Batch(s, 7)
    b.write_all(wl.state, wl.pars, np.zeros(7), np.zeros(7))
    g = np.linspace(0.0, 1.0, 5)[:, None] * np.where(np.arange(7) % 2 == 0, 1.0, -1.0)
    b.propagate_grid(g)
    b.write_all(wl.state, wl.pars, np.zeros(7), np.zeros(7))
    bad = g.copy()
    bad[row, col] = bad[row - 1, col] if row else 0.5
    with pytest.raises(_lib.HyxError, match=msg + f".*instance {col}|instance {col}.*" + msg):
        b.propagate_grid(bad)


def test_device_pointer_of_a_filled_batch():
    # From its second fill on a small batch returns before its copy ends; the device pointer waits
    # for it, so that any stream reads the new values.
    H = _hip()
    n = 501
    wl = workloads.cr3bp(n)
    b = _lib.Batch(_lib.System(hy.taylor_decompose(wl.sys), 19), n)
    for rep in range(4):
        st = wl.state + rep
        b.write_all(st, wl.pars, np.full(n, float(rep)), np.zeros(n))
        out = np.empty_like(st)
        assert H.hipMemcpy(out.ctypes.data, b.device_ptr(_lib.FIELD_STATE), out.nbytes, D2H) == 0
        assert np.array_equal(out, st)
