"""CG solves as one cooperative launch (messages between the iteration
steps) against the two-launches-per-iteration form: the same iterates, so
the same results bit for bit and the same iteration counts, for the pressure
solve (pressure.py:67-112) and the implicit diffusion solve
(diffusion.py:137-167)."""
import functools

import numpy as np
import pytest
import torch

from oracle import initial_conditions as oic
from oracle.grid_ops import Grid as OGrid

pytestmark = pytest.mark.gpu
TWO_PI = 2 * np.pi


def _dev():
  return torch.device('cuda', 0)


def _cfd():
  import jax_cfd_amd.base as cfd
  return cfd


def _grid(n):
  return _cfd().grids.Grid((n, n), domain=((0, TWO_PI), (0, TWO_PI)))


def _state(n, seed, vmax):
  cfd = _cfd()
  og = OGrid.from_domain((n, n), ((0, TWO_PI), (0, TWO_PI)))
  v0 = oic.filtered_velocity_field(seed, og, vmax, 4)
  bc = cfd.boundaries.periodic_boundary_conditions(2)
  return tuple(cfd.grids.GridVariable(cfd.grids.GridArray(
      torch.as_tensor(u.data, device=_dev()), u.offset, _grid(n)), bc) for u in v0)


@pytest.mark.parametrize("n", [64, 256, 512])
def test_pressure_cg_persistent_equals_two_kernel_form(n):
  cfd = _cfd()
  grid = _grid(n)
  dt = cfd.equations.stable_time_step(7.0, 0.5, 1e-3, grid)
  solve = functools.partial(cfd.pressure.solve_cg, rtol=1e-6, atol=1e-6)
  step = cfd.equations.semi_implicit_navier_stokes(
      1.0, 1e-3, dt, grid,
      convect=lambda v: tuple(cfd.advection.advect_van_leer(u, v, dt) for u in v),
      forcing=cfd.forcings.simple_turbulence_forcing(grid, 1.0, 4, -0.1, 'kolmogorov'),
      pressure_solve=solve)
  state = _state(n, 3, 7.0)
  runs = []
  for persistent in (True, False):
    step.plan().set_cg_persistent(persistent)
    print(f"pressure CG n={n} persistent={persistent}: 3 steps", flush=True)
    out = cfd.funcutils.repeated(step, 3)(state)
    torch.cuda.synchronize()
    runs.append(([u.data.clone() for u in out], step.plan().cg_iterations))
  step.plan().set_cg_persistent(False)
  (a, ka), (b, kb) = runs
  print(f"  iterations of the last step: {ka} (one launch), {kb} (two per iteration)")
  assert ka == kb and ka > 0
  for x, y in zip(a, b):
    assert torch.equal(x, y)


@pytest.mark.parametrize("n", [64, 256])
def test_diffusion_cg_persistent_equals_two_kernel_form(n):
  cfd = _cfd()
  from jax_cfd_amd import _lib
  from jax_cfd_amd.base import _fvm
  grid = _grid(n)
  rng = np.random.default_rng(7)
  bc = cfd.boundaries.periodic_boundary_conditions(2)
  state = tuple(cfd.grids.GridVariable(cfd.grids.GridArray(
      torch.as_tensor(rng.standard_normal((n, n)).astype(np.float32), device=_dev()), o, grid), bc)
      for o in grid.cell_faces)
  plan = _fvm.plan_for(_fvm.spec_from_grid(
      grid, dt=0.02, viscosity=0.05, diffusion=_lib.DIFFUSION_IMPLICIT_CG,
      **cfd.diffusion.cg_spec_fields(rtol=1e-7, atol=1e-6)), _dev())
  runs = []
  for persistent in (True, False):
    plan.set_cg_persistent(persistent)
    print(f"diffusion CG n={n} persistent={persistent}", flush=True)
    out = cfd.diffusion.solve_cg(state, 0.05, 0.02, rtol=1e-7, atol=1e-6)
    torch.cuda.synchronize()
    runs.append(([u.data.clone() for u in out],
                 [plan.diffusion_cg_iterations(m) for m in range(2)]))
  plan.set_cg_persistent(False)
  (a, ka), (b, kb) = runs
  print(f"  iterations per component: {ka} (one launch), {kb} (two per iteration)")
  assert ka == kb and min(ka) > 0
  for x, y in zip(a, b):
    assert torch.equal(x, y)
