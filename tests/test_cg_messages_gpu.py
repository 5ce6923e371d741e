"""The one-launch CG solve at the row counts its own test leaves out, cut off
by maxiter, from two threads at once, and given up: bit for bit the two-kernel
form."""
import functools
import threading

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


def test_two_threads():
  # each thread steps its own plan on its own stream; the calls release the
  # interpreter, so their solves are under way together
  steps = [_step(128, rtol=1e-6, atol=1e-6), _step(256, rtol=1e-5, atol=1e-6)]
  states = [cg._state(128, 3, 7.0), cg._state(256, 4, 7.0)]
  alone = [_run(s, x, False, 12)[0] for s, x in zip(steps, states)]
  repeated, start, out = cg._cfd().funcutils.repeated, threading.Barrier(2), [None, None]
  torch.cuda.synchronize()

  def work(k):
    with torch.cuda.stream(torch.cuda.Stream()):
      start.wait(30)
      out[k] = repeated(steps[k], 12)(states[k])
      torch.cuda.current_stream().synchronize()

  threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
  for t in threads:
    t.start()
  for t in threads:
    t.join()
  for got, want in zip(out, alone):
    for x, y in zip(got, want):
      assert torch.equal(x.data, y)


@pytest.mark.parametrize('n', [64, 256, 512])
def test_given_up_pressure_solve(n):
  # a host-side limit of no polls: every workgroup gives up at its first message
  step, state = _step(n, rtol=1e-6, atol=1e-6), cg._state(n, 3, 7.0)
  plan = step.plan()
  want, iterations = _run(step, state, False, 3)
  before = plan.cg_solves
  plan.set_cg_polls(0)
  got, its = _run(step, state, True, 3)
  after = plan.cg_solves
  plan.set_cg_polls(1 << 20)
  assert its == iterations
  for x, y in zip(got, want):
    assert torch.equal(x, y)
  # one wait, then two launches per iteration without another
  assert {k: after[k] - before[k] for k in after} == {'one_launch': 0, 'two_launches': 3, 'given_up': 1}
  got, its = _run(step, state, True, 3)
  assert its == iterations and plan.cg_solves['one_launch'] == after['one_launch'] + 3
  for x, y in zip(got, want):
    assert torch.equal(x, y)


@pytest.mark.parametrize('n', [64, 256])
def test_given_up_diffusion_solve(n):
  cfd = cg._cfd()
  from jax_cfd_amd import _lib
  from jax_cfd_amd.base import _fvm
  grid, bc = cg._grid(n), cfd.boundaries.periodic_boundary_conditions(2)
  gen = torch.Generator(device=cg._dev()).manual_seed(n)
  state = tuple(cfd.grids.GridVariable(cfd.grids.GridArray(
      torch.randn((n, n), device=cg._dev(), generator=gen), o, grid), bc) for o in grid.cell_faces)
  plan = _fvm.plan_for(_fvm.spec_from_grid(
      grid, dt=0.02, viscosity=0.04, diffusion=_lib.DIFFUSION_IMPLICIT_CG,
      **cfd.diffusion.cg_spec_fields(rtol=1e-7, atol=1e-6)), cg._dev())
  runs = []
  for persistent, polls in ((False, 1 << 20), (True, 0)):
    plan.set_cg_persistent(persistent)
    plan.set_cg_polls(polls)
    before = plan.cg_solves
    out = cfd.diffusion.solve_cg(state, 0.04, 0.02, rtol=1e-7, atol=1e-6)
    torch.cuda.synchronize()
    runs.append(([u.data.clone() for u in out], [plan.diffusion_cg_iterations(m) for m in range(2)],
                 {k: x - before[k] for k, x in plan.cg_solves.items()}))
  plan.set_cg_polls(1 << 20)
  (a, ka, ca), (b, kb, cb) = runs
  assert ka == kb and min(ka) > 0
  assert ca == {'one_launch': 0, 'two_launches': 2, 'given_up': 0}
  assert cb == {'one_launch': 0, 'two_launches': 2, 'given_up': 1}  # the first component's
  for x, y in zip(a, b):
    assert torch.equal(x, y)
