"""Explicit kernels of more than 16 states in registers against the private
segment: the same results bit for bit in the parity build, below, at and past
the point where registers run out."""

import numpy as np
import pytest

import cubie_amd as ca

pytestmark = pytest.mark.gpu


def _ring(n, precision):
    eqs = [f"dx{i} = (x{(i + 1) % n} - x{(i - 2) % n})*x{(i - 1) % n} - x{i} + F" for i in range(n)]
    return ca.create_ODE_system(eqs, states={f"x{i}": 8.0 for i in range(n)},
                                parameters={"F": 8.0}, precision=precision, name=f"lorenz96_{n}")


@pytest.mark.parametrize("n,precision,algorithm", [
    (17, np.float64, "dormand-prince-54"), (32, np.float64, "dormand-prince-54"),
    (39, np.float64, "dormand-prince-54"), (60, np.float32, "dormand-prince-54"),
    (24, np.float64, "rk4")])
def test_registers_match_the_private_segment(n, precision, algorithm):
    rng = np.random.default_rng(n)
    runs = 200
    inits = (8.0 + rng.normal(0.0, 1.0, (n, runs))).astype(precision)
    params = rng.uniform(7.0, 9.0, (1, runs)).astype(precision)
    kw = dict(dt=2.0 ** -7) if algorithm == "rk4" else dict(atol=1e-6, rtol=1e-5)

    def solver(placement):
        return ca.Solver(_ring(n, precision), algorithm=algorithm, save_every=0.0625,
                         output_types=["state", "time"], buffer_placement=placement,
                         deterministic_pow=True, **kw)

    solver("memory").kernel.compile_only(0.5)
    a = solver("auto")
    assert a.kernel.spec_for(0.5).resolved_placement == "registers"
    res = [s.solve(inits, params, duration=0.5) for s in (a, solver("memory"))]
    assert np.all(res[0].status_codes == 0)
    assert np.array_equal(res[0].status_codes, res[1].status_codes)
    assert np.array_equal(res[0].state, res[1].state)
