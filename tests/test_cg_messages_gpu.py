"""The one-launch CG solve at the row counts its own test leaves out, cut off
by maxiter, and from two streams at once: bit for bit the two-kernel form."""
import functools

import pytest
import torch

import test_cg_persistent_gpu as cg

pytestmark = pytest.mark.gpu


def _step(n, **solve):
  cfd = cg._cfd()
  grid = cg._grid(n)
  dt = cfd.equations.stable_time_step(7.0, 0.5, 1e-3, grid)
  return cfd.equations.semi_implicit_navier_stokes(
      1.0, 1e-3, dt, grid,
      convect=lambda v: tuple(cfd.advection.advect_van_leer(u, v, dt) for u in v),
      forcing=cfd.forcings.simple_turbulence_forcing(grid, 1.0, 4, -0.1, 'kolmogorov'),
      pressure_solve=functools.partial(cfd.pressure.solve_cg, **solve))


def _run(step, state, persistent, steps):
  step.plan().set_cg_persistent(persistent)
  out = cg._cfd().funcutils.repeated(step, steps)(state)
  torch.cuda.synchronize()
  step.plan().set_cg_persistent(True)
  return [u.data.clone() for u in out], step.plan().cg_iterations


@pytest.mark.parametrize('n,solve', [(32, dict(rtol=1e-6, atol=1e-6)), (128, dict(rtol=1e-5, atol=1e-6)),
                                     (1024, dict(rtol=1e-2, atol=1e-3)),
                                     (256, dict(rtol=1e-7, atol=1e-8, maxiter=5)),
                                     (64, dict(rtol=1e9, atol=1e-6))])  # converged at once
def test_one_launch_equals_two_per_iteration(n, solve):
  step, state = _step(n, **solve), cg._state(n, 3, 7.0)
  (a, ka), (b, kb) = (_run(step, state, persistent, 3) for persistent in (True, False))
  assert ka == kb and ka == solve.get('maxiter', ka)
  for x, y in zip(a, b):
    assert torch.equal(x, y)


def test_two_streams():
  steps = [_step(128, rtol=1e-6, atol=1e-6), _step(256, rtol=1e-5, atol=1e-6)]
  states = [cg._state(128, 3, 7.0), cg._state(256, 4, 7.0)]
  alone = [_run(s, x, False, 2)[0] for s, x in zip(steps, states)]
  streams = [torch.cuda.Stream() for _ in steps]
  torch.cuda.synchronize()
  out = []
  for step, state, stream in zip(steps, states, streams):
    with torch.cuda.stream(stream):
      out.append(cg._cfd().funcutils.repeated(step, 2)(state))
  torch.cuda.synchronize()
  for got, want in zip(out, alone):
    for x, y in zip(got, want):
      assert torch.equal(x.data, y)
