"""propagate_grid of the unrolled form (grid points evaluated inside the step, from registers):
batch sizes around a wavefront, one to many points per step, per-instance grids in either
direction, early ends, against the oracle."""

import numpy as np
import pytest

import heyoka_amd as hy
import pyoracle as O
from heyoka_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["persistent", "plain"])
@pytest.mark.parametrize("N,npts,limit", [(1, 1, 0), (1, 300, 0), (63, 2, 0), (65, 40, 0), (200, 40, 3), (130, 7, 1)])
def test_dense_grid_vs_oracle(N, npts, limit, mode):
    print(f"[gpu] dense grid N={N} npts={npts} limit={limit} {mode}", flush=True)
    wl = W.cr3bp(N)
    rng = np.random.default_rng(N)
    end = rng.uniform(1.0, 6.0, N) * np.where(np.arange(N) % 3 == 1, -1.0, 1.0)
    grid = np.ascontiguousarray(np.linspace(0.0, 1.0, npts)[:, None] * end)
    ta = hy.taylor_adaptive_batch(wl.sys, wl.state, pars=wl.pars, tol=1e-15, gpu_mode=mode)
    assert ta.code_form == "unrolled"
    _, out = ta.propagate_grid(grid, max_steps=limit)
    r = O.propagate_grid(hy.taylor_decompose(wl.sys), 19, wl.state, grid, pars=wl.pars, max_steps=limit)
    assert np.array_equal(np.isnan(out), np.isnan(r["out"]))
    ok = ~np.isnan(out)
    np.testing.assert_allclose(out[ok], r["out"][ok], rtol=1e-9, atol=1e-9)
    assert np.array_equal(out[0], wl.state) and [x[3] for x in ta.propagate_res] == list(r["nsteps"])


def test_dense_grid_stops_at_a_non_finite_state():
    # Instance 1 starts on a primary: its points stay NaN, the other's do not.
    wl = W.cr3bp(2)
    st = wl.state.copy()
    st[:2, 1] = [-wl.pars[0, 1], 0.0]
    ta = hy.taylor_adaptive_batch(wl.sys, st, pars=wl.pars, tol=1e-15)
    _, out = ta.propagate_grid(np.repeat(np.linspace(0.0, 2.0, 9)[:, None], 2, axis=1))
    assert int(ta.propagate_res[1][0]) == int(hy.taylor_outcome.err_nf_state)
    assert np.isnan(out[1:, :, 1]).all() and np.isfinite(out[:, :, 0]).all()
