"""The adjoint with a checkpoint at every step against the one that replays
segments: the same gradients to rounding, at batch sizes around a wavefront,
with runs of different lengths, saved rows, every differentiable summary, both
families and precisions; and a first tape that turns out too short."""

import numpy as np
import pytest

import cubie_amd as ca
from cubie_amd.batchsolving import adjoint as adj
from cubie_amd.runtime import kcache
from systems import hh_batch, hh_driver, hodgkin_huxley, lorenz, lorenz_batch

pytestmark = pytest.mark.gpu


def _grads(solver, inits, params, duration, every, seed=5):
    import torch
    rec = adj.record(solver.kernel, inits, params, duration=duration, checkpoint_every=every)
    out = rec.outputs
    assert int(out.status_codes.abs().sum()) == 0
    gen = torch.Generator().manual_seed(seed)
    draw = lambda x: torch.randn(tuple(x.shape), generator=gen, dtype=torch.float64)
    gs = draw(out.state) if out.state.ndim == 3 else None
    gss = draw(out.state_summaries) if out.state_summaries.ndim == 3 else None
    gi, gp, _ = adj.backward(rec, gs, gss)
    return rec, np.concatenate([gi.cpu().numpy(), gp.cpu().numpy()]).astype(np.float64)


def _compare(solver, inits, params, duration, bar):
    spec = solver.kernel.spec_for(duration, False, adjoint=True, adj_ckpt_every=7)
    kcache.get_code(spec.source(), spec.compile_options())
    every, a = _grads(solver, inits, params, duration, 32)
    segments, b = _grads(solver, inits, params, duration, 7)
    assert every.checkpoint_every == 1 and segments.checkpoint_every == 7
    assert every.max_steps == segments.max_steps
    err = np.abs(a - b).max(axis=0) / np.abs(b).max(axis=0)
    assert err.max() <= bar, err.max()
    return every


def _hh(alg, **kw):
    s = ca.Solver(hodgkin_huxley(np.float64), algorithm=alg, atol=1e-6, rtol=1e-6, save_every=2.5,
                  summarise_every=5.0, sample_summaries_every=0.25, summarise_variables=["V", "h"],
                  output_types=["state", "mean", "max", "rms"], deterministic_pow=True, **kw)
    s._configure_drivers(hh_driver())
    return s


@pytest.mark.parametrize("n", [1, 63, 65, 300])
@pytest.mark.parametrize("alg", ["dormand-prince-54", "tsit5"])
def test_hodgkin_huxley(alg, n):
    """Adaptive FP64 steps, so lanes end at different steps. The parity
    build's forward passes are the same bit for bit; the two orders of
    evaluation of the backward pass differ by rounding alone: 2e-16 x about 20
    operations x 300 steps, and a cancellation of up to 1e3 in the sums over
    the spikes of 20 ms, 1.3e-9."""
    inits, params = hh_batch(n, seed=70)
    _compare(_hh(alg), inits, params, 20.0, 1e-8)


def test_rosenbrock_runs_do_not_depend_on_their_neighbours():
    """Each run's gradient in a batch past one wavefront is the one it has
    alone, bit for bit. (Rosenbrock segments are not a reference to rounding:
    their replay solves the stages directly where the forward pass iterates to
    its Krylov tolerance. Central differences check the gradient itself.)"""
    import torch
    inits, params = hh_batch(65, seed=73)
    s = _hh("ros3p", linear_correction_type="bicgstab")

    def grads(pick):
        rec = adj.record(s.kernel, inits[:, pick], params[:, pick], duration=20.0)
        assert rec.checkpoint_every == 1
        gi, gp, _ = adj.backward(rec, torch.ones_like(rec.outputs.state),
                                 torch.ones_like(rec.outputs.state_summaries))
        return np.concatenate([gi.cpu().numpy(), gp.cpu().numpy()])

    whole = grads(np.arange(65))
    assert np.isfinite(whole).all() and np.abs(whole).max() > 0
    for i in (0, 40, 64):
        assert np.array_equal(grads(np.array([i]))[:, 0], whole[:, i])


def test_fp32_lorenz():
    inits, params = lorenz_batch(130, seed=71)
    s = ca.Solver(lorenz(np.float32), algorithm="dormand-prince-54", atol=1e-5, rtol=1e-4,
                  save_every=0.125, output_types=["state"], deterministic_pow=True)
    _compare(s, inits.astype(np.float32), params.astype(np.float32), 1.0, 2e-3)


def test_first_tape_too_short(monkeypatch):
    inits, params = lorenz_batch(100, seed=72)
    s = ca.Solver(lorenz(np.float64), algorithm="dormand-prince-54", atol=1e-8, rtol=1e-6,
                  save_every=0.01, output_types=["state"])
    rec, a = _grads(s, inits, params, 2.0, 32)
    assert rec.max_steps > 150
    monkeypatch.setattr(adj, "TAPE_FIRST_TRY", 100 * 41 * 100)
    rec2, b = _grads(s, inits, params, 2.0, 32)
    assert rec2.max_steps == rec.max_steps and np.array_equal(a, b)


def test_tape_is_freed_with_its_graph():
    """No reference cycle keeps a tape once its outputs are gone."""
    import gc
    import torch
    inits, params = lorenz_batch(64, seed=74)
    s = ca.Solver(lorenz(np.float64), algorithm="dormand-prince-54", atol=1e-8, rtol=1e-6,
                  save_every=0.01, output_types=["state"])
    x = torch.tensor(inits, requires_grad=True)
    p = torch.tensor(params)

    def once():
        state, _, _ = ca.solve_adjoint(s, x, p, duration=2.0)
        state.sum().backward()

    once()
    torch.cuda.synchronize()
    gc.collect()
    gc.disable()
    try:
        before = torch.cuda.memory_allocated()
        for _ in range(3):
            once()
        assert torch.cuda.memory_allocated() == before
    finally:
        gc.enable()
