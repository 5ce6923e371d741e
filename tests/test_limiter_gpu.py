"""The limiter's quotient and sign forms on differences that smooth fields do
not have: flat, signed-zero, one-cell jumps over many scales, and infinities
and NaN, explicit terms against the fp32 oracle."""
import numpy as np
import pytest
import torch

import test_fvm_gpu as fvm

pytestmark = pytest.mark.gpu


def _fields(kind, n):
  rng = np.random.default_rng(11)
  x = rng.standard_normal((2, n, n))
  if kind == 'flat':
    x = np.where(rng.random((2, n, n)) < 0.5, 0.5, np.where(rng.random((2, n, n)) < 0.5, 0.0, -0.0))
  elif kind == 'scales':  # differences of 1e-12 beside differences of 1
    x = 1.0 + x * 10.0 ** rng.integers(-12, 1, (2, n, n))
  elif kind == 'tiny':  # all differences near the smallest normal number
    x = x * 1e-36
  elif kind == 'large':
    x = x * 1e15
  elif kind == 'wild':
    x[0, 5, 7], x[1, 20, 30], x[0, 40, 41] = np.inf, -np.inf, np.nan
  return x.astype(np.float32)


@pytest.mark.parametrize('kind', ['flat', 'scales', 'tiny', 'large', 'wild'])
@pytest.mark.parametrize('n', [64, 256])
def test_explicit_terms_of_uneven_fields(kind, n):
  # the terms round in the oracle's order, some ten times each: 1e-6 of the
  # largest; the same cells are not finite (an infinite difference over the grid
  # step is NaN in the kernels, over_step, and infinite in the oracle)
  ogrid, v0, dt, ostep, step = fvm._config(n, 3, 1.0, False)
  x = _fields(kind, n)
  v = tuple(type(c)(d, c.offset) for c, d in zip(v0, x))
  cfd = fvm._cfd()
  et = cfd.equations.navier_stokes_explicit_terms(
      1.0, 1e-3, dt, fvm._grid(n), convect=lambda v: tuple(cfd.advection.advect_van_leer(u, v, dt) for u in v))
  with np.errstate(all='ignore'):
    want = ostep.explicit_terms(v)
  for g, w in zip(et(fvm._state(v, n)), want):
    g, w = g.data.cpu().numpy(), w.data
    ok = np.isfinite(w)
    assert np.array_equal(np.isfinite(g), ok)
    assert np.abs(g[ok] - w[ok]).max() <= 1e-6 * np.abs(w[ok]).max()


@pytest.mark.parametrize('n,batch', [(256, 32), (512, 8)])
def test_marching_rows_of_uneven_fields(n, batch):
  import test_launch_shapes_gpu as shapes
  plan, u, v = shapes._fvm(n, batch)
  for b, kind in enumerate(['flat', 'scales', 'tiny', 'large']):
    u[b], v[b] = (torch.as_tensor(x).cuda() for x in _fields(kind, n))
  got = plan.step(u, v, 1)
  plan.set_tiles(1, 1, 1, 8)
  want = plan.step(u, v, 1)
  assert plan.tiles['rows_forward'] == 1
  for g, w in zip(got, want):
    assert torch.allclose(g, w, rtol=0, atol=0, equal_nan=True)  # the large fields overflow


def _huge(kind, n):
  """u of one size and alternating sign along x, so that the faces between
  carry no u and the terms of u stay finite; v = 0.01 along y."""
  x = np.ones((2, n, n))
  sign = np.where(np.arange(n) % 2, -1.0, 1.0)[:, None]
  y = np.arange(n)[None, :]
  if kind == 'beyond 2^126':  # differences of 4e37 to 1e38, sums beyond 2^126
    x[0] = sign * 1e38 * np.sin(2 * np.pi * (y + 0.3) / 8)
  elif kind == 'infinite sum':  # differences of 3e38 along x
    x[0] = sign * 1.5e38
  elif kind == 'subnormal':  # differences and their sums below 2^-126
    x[0] = sign * np.random.default_rng(5).integers(1, 2 ** 21, (n, n)) * 2.0 ** -149
  x[1] = 0.01
  return x.astype(np.float32)


@pytest.mark.parametrize('kind', ['beyond 2^126', 'infinite sum', 'subnormal'])
@pytest.mark.parametrize('n', [64, 256])
def test_explicit_terms_beyond_the_quotients_range(kind, n):
  # as above, without viscosity (differences of differences overflow); the
  # subnormal terms carry the fields' own spacing, some ten roundings to 2^-149
  # over the grid step
  ogrid, v0, dt, _, _ = fvm._config(n, 3, 1.0, False)
  ostep = fvm.ofvm.FVMStep(ogrid, dt=dt, viscosity=None, forcing=None)
  x = _huge(kind, n)
  v = tuple(type(c)(d, c.offset) for c, d in zip(v0, x))
  cfd = fvm._cfd()
  et = cfd.equations.navier_stokes_explicit_terms(
      1.0, None, dt, fvm._grid(n), convect=lambda v: tuple(cfd.advection.advect_van_leer(u, v, dt) for u in v))
  with np.errstate(all='ignore'):
    want = ostep.explicit_terms(v)[0].data
  got = et(fvm._state(v, n))[0].data.cpu().numpy()
  assert np.isfinite(want).all() and np.isfinite(got).all()
  floor = 10 * 2.0 ** -149 * n / (2 * np.pi)
  assert np.abs(got - want).max() <= max(1e-6 * np.abs(want).max(), floor)
