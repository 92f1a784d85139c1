"""The occupancy floor a batch's kernel is compiled with (no GPU: the register
count comes from the code object's metadata)."""

import numpy as np

import cubie_amd as ca
from cubie_amd.batchsolving import kernel as bk
from cubie_amd.runtime import kcache
from systems import hodgkin_huxley, lorenz


def test_register_count_of_a_code_object():
    solver = ca.Solver(lorenz(np.float64), algorithm="tsit5", save_every=0.5,
                       output_types=["state"])
    code = solver.kernel.compile_only(1.0)
    for name in ("cubie_integrate", "cubie_integrate_persistent"):
        assert 16 <= kcache.vgpr_count(code, name) <= 512
    assert kcache.vgpr_count(code, "cubie_adjoint") is None


def test_floor_only_where_a_second_wavefront_waits(monkeypatch):
    monkeypatch.setattr(bk, "_compute_units", lambda: 256)
    solver = ca.Solver(hodgkin_huxley(np.float64), algorithm="l_stable_dirk_3", dt=2.0 ** -6,
                       linear_correction_type="bicgstab", save_every=1.0, output_types=["state"])
    k = solver.kernel
    for regs, n_runs, floor in ((301, 65536, 0), (301, 65537, 2), (512, 10 ** 6, 2),
                                (256, 10 ** 6, 0), (None, 10 ** 6, 0)):
        monkeypatch.setattr(kcache, "vgprs_of_parts", lambda *a, regs=regs: regs)
        assert k.launch_spec(n_runs, 1.0).waves_per_eu == floor
    k.update({"waves_per_eu": 1})
    monkeypatch.setattr(kcache, "vgprs_of_parts", lambda *a: 301)
    assert k.launch_spec(10 ** 6, 1.0).waves_per_eu == 1


def test_explicit_kernels_keep_their_registers(monkeypatch):
    monkeypatch.setattr(bk, "_compute_units", lambda: 256)
    monkeypatch.setattr(kcache, "vgprs_of_parts", lambda *a: 333)
    solver = ca.Solver(lorenz(np.float64), algorithm="tsit5", save_every=0.5,
                       output_types=["state"])
    assert solver.kernel.launch_spec(10 ** 6, 1.0).waves_per_eu == 0


def _chain(n, precision):
    return ca.create_ODE_system([f"dx{i} = x{(i + 1) % n} - p*x{i}" for i in range(n)],
                                states={f"x{i}": 1.0 for i in range(n)}, parameters={"p": 2.0},
                                precision=precision, name=f"chain{n}")


def test_placement_of_explicit_kernels():
    """Registers up to 640 words of vectors; implicit kernels, the adjoint and
    an explicit choice as before."""
    for n, precision, alg, want in ((16, np.float64, "dormand-prince-54", "registers"),
                                    (39, np.float64, "dormand-prince-54", "registers"),
                                    (41, np.float64, "dormand-prince-54", "memory"),
                                    (41, np.float32, "dormand-prince-54", "registers"),
                                    (41, np.float64, "rk4", "registers"),
                                    (17, np.float64, "ros3p", "memory")):
        k = ca.Solver(_chain(n, precision), algorithm=alg, save_every=0.5,
                      output_types=["state"]).kernel
        assert k.spec_for(1.0).resolved_placement == want, (n, precision, alg)
        if alg != "ros3p":
            k.update({"buffer_placement": "memory"})
            assert k.spec_for(1.0).resolved_placement == "memory"
    k = ca.Solver(_chain(20, np.float64), algorithm="tsit5", save_every=0.5,
                  output_types=["state"]).kernel
    assert k.spec_for(1.0, adjoint=True).resolved_placement == "memory"
