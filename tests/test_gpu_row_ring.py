"""Per-row outputs of adaptive runs through the plain kernel's LDS row ring:
the same arrays, bit for bit, as the parity build writes directly, at batch
sizes around a wavefront and a workgroup, with every kind of row, rows that
outnumber the ring many times over, and runs that end early."""

import numpy as np
import pytest

import cubie_amd as ca
from systems import lorenz, lorenz_batch, robertson, robertson_batch

pytestmark = pytest.mark.gpu


def decay(precision):
    return ca.create_ODE_system(
        ["dx = -k*x + 0.1*y*y", "dy = k*x - y*y", "e = x + y", "q = x - y"],
        states={"x": 1.0, "y": 0.5}, parameters={"k": 1.0}, observables=["e", "q"],
        precision=precision, name="decay2")


def _solver(make, staging):
    solver = make()
    solver.kernel.update({"output_staging": staging})
    return solver


def _solve(make, inits, params, duration, staging):
    solver = _solver(make, staging)
    assert (solver.kernel.row_ring() > 0) == (staging == "auto")
    res = solver.solve(inits, params, duration=duration, nan_error_trajectories=False)
    return {k: getattr(res, k) for k in ("state", "observables", "iteration_counters",
                                         "status_codes")}


def _same(make, inits, params, duration):
    _solver(make, "direct").kernel.compile_only(duration)
    a = _solve(make, inits, params, duration, "auto")
    b = _solve(make, inits, params, duration, "direct")
    for k in a:
        assert (a[k] is None) == (b[k] is None), k
        if a[k] is not None:
            assert a[k].shape == b[k].shape and np.array_equal(a[k], b[k]), k
    return a


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 1000])
def test_states_and_time(n):
    inits, params = lorenz_batch(n, seed=5)
    make = lambda: ca.Solver(lorenz(np.float64), algorithm="dormand-prince-54", atol=1e-8,
                             rtol=1e-6, save_every=0.01, output_types=["state", "time"],
                             deterministic_pow=True)
    out = _same(make, inits, params, 0.5)
    assert np.all(out["status_codes"] == 0) and np.all(out["state"][:, 2].any(axis=1))


@pytest.mark.parametrize("precision", [np.float32, np.float64])
def test_observables_and_counters(precision):
    rng = np.random.default_rng(6)
    n = 321
    params = rng.uniform(0.1, 40.0, (1, n))
    inits = rng.uniform(0.1, 2.0, (2, n))
    make = lambda: ca.Solver(decay(precision), algorithm="tsit5", atol=1e-6, rtol=1e-5,
                             save_every=0.125, deterministic_pow=True,
                             output_types=["state", "observables", "time",
                                           "iteration_counters"])
    _same(make, inits, params, 4.0)


def test_save_table_and_runs_that_end_early():
    """Robertson on a save table; with dt_min at 1e-3 the early steps of most
    runs fall below it and the run ends, leaving zero rows."""
    inits, params = robertson_batch(130, seed=7)
    params[:, ::3] *= np.array([[1.0], [1e-6], [1e-3]])
    table = np.logspace(-3.0, 1.0, 37)
    table[-1] = 10.0
    make = lambda: ca.Solver(robertson(np.float64), algorithm="ros3p", atol=1e-10, rtol=1e-6,
                             dt=1e-2, dt_min=1e-3, linear_correction_type="bicgstab",
                             save_times=table, output_types=["state"], deterministic_pow=True)
    out = _same(make, inits, params, 10.0)
    ended = out["status_codes"] != 0
    assert ended.any() and not ended.all()
    assert np.all(out["state"][-1][:, ended] == 0.0)
    assert np.all(out["state"][-1][:, ~ended].sum(axis=0) > 0.5)


@pytest.mark.parametrize("n", [1, 63, 65, 257])
def test_final_state_alone_is_written_in_place(n):
    """Two rows a run and no save grid: the plain kernel writes them directly,
    the same as the persistent kernel's staged and transposed ones."""
    inits, params = lorenz_batch(n, seed=8)

    def make(mode):
        return ca.Solver(lorenz(np.float64), algorithm="dormand-prince-54", atol=1e-8,
                         rtol=1e-6, output_types=["state", "time"], deterministic_pow=True,
                         kernel_mode=mode)
    a, b = make("plain"), make("persistent")
    assert a.kernel.row_ring() == 0 and not a.kernel.run_major_rows()
    assert b.kernel.run_major_rows()
    ra, rb = (s.solve(inits, params, duration=0.5) for s in (a, b))
    assert ra.state.shape == rb.state.shape and ra.state.shape[0] == 2
    assert np.array_equal(ra.state, rb.state) and np.all(ra.status_codes == 0)
