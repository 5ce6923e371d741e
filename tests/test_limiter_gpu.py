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
