"""The tower's convolutions against 64-bit ones: rounding, and values whose
three-part split does not exist."""
import numpy as np
import pytest
import torch

import test_ml_gpu as ml

pytestmark = pytest.mark.gpu


def _conv(x, w, b):
  x = torch.nn.functional.pad(x, (1, 1, 1, 1), mode='circular')
  return torch.nn.functional.conv2d(x, torch.as_tensor(np.asarray(w, np.float64)).permute(3, 2, 0, 1),
                                    torch.as_tensor(np.asarray(b, np.float64)))


def _tower(u, v, params):
  x = torch.stack([u, v]).double().cpu()[None]
  for k, (w, b) in enumerate(params):
    x = _conv(x, w, b)
    if k + 1 < len(params):
      x = torch.fmax(x, torch.zeros_like(x))
  return x[0]


@pytest.mark.parametrize('n', [32, 64])
@pytest.mark.parametrize('hidden', [16, 32, 64])
def test_tower_rounding(n, hidden):
  # A layer rounds each sum at most 18 times (rms 2^-24 / sqrt(3) of the sum
  # each) and once for the bias: three layers stay under 8 x 2^-24 of the
  # output, rms.  One part product left out is 1e-6 and more.
  params, v0 = ml._case(n, hidden, 2, seed=3)
  plan = ml._model(n, params, hidden, 2)[0].plan(ml._dev())
  u, v = (torch.as_tensor(x.data, device=ml._dev()) for x in v0)
  got = plan.tower(u, v, coefficients=False)[0, :120].double().cpu()
  want = _tower(u, v, params)
  assert float((got - want).norm() / want.norm()) <= 2.0 ** -21


@pytest.mark.parametrize('hidden', [16, 32, 64])
@pytest.mark.parametrize('value', [2.5e38, 1.7e38, float('inf'), float('nan')])
def test_tower_values_without_a_split(hidden, value):
  # the first layer passes u on in its first channel; the cell is a corner, so
  # that the periodic halos of four workgroups hold it
  n = 64
  params, v0 = ml._case(n, hidden, 2, seed=3)
  w0 = np.zeros_like(params[0][0])
  w0[1, 1, 0, 0] = 1.0
  w0[1, 1, 1, 1:] = 1.0
  params[0] = (w0, np.zeros_like(params[0][1]))
  params[1] = (params[1][0] * np.float32(0.25), params[1][1])
  plan = ml._model(n, params, hidden, 2)[0].plan(ml._dev())
  u, v = (torch.as_tensor(x.data, device=ml._dev()).clone() for x in v0)
  u[0, 0] = value
  got = plan.tower(u, v, coefficients=False)[0, :120].double().cpu()
  want = _tower(u, v, params)
  far = torch.ones(n, n, dtype=torch.bool)
  far[[-2, -1, 0, 1, 2]] = False
  far |= ~torch.roll(torch.arange(n) < 5, -2)
  assert torch.isfinite(got[:, far]).all()
  for g, w in ((got[:, far], want[:, far]), (got[:, ~far], want[:, ~far])):
    assert torch.equal(torch.isnan(g), torch.isnan(w))
    assert torch.equal(torch.isinf(g), torch.isinf(w))
    ok = torch.isfinite(w)
    if ok.any():
      assert float((g[ok] - w[ok]).abs().max()) <= 1e-5 * float(w[ok].abs().max())


@pytest.mark.parametrize('hidden', [16, 32, 64])
@pytest.mark.parametrize('scale', [1e-35, 1e-30])
def test_tower_rounding_of_small_values(hidden, scale):
  # as test_tower_rounding, on activations near and under the least ones whose
  # three bf16 parts are normal numbers; no biases, which would cover them
  n = 64
  params, v0 = ml._case(n, hidden, 2, seed=3)
  params = [(w, np.zeros_like(b)) for w, b in params]
  plan = ml._model(n, params, hidden, 2)[0].plan(ml._dev())
  u, v = (torch.as_tensor(x.data, device=ml._dev()) * scale for x in v0)
  got = plan.tower(u, v, coefficients=False)[0, :120].double().cpu()
  want = _tower(u, v, params)
  assert float((got - want).norm() / want.norm()) <= 2.0 ** -21


@pytest.mark.parametrize('n,hidden,layers', [(256, 64, 6), (128, 32, 3), (64, 16, 2)])
def test_values_without_a_split_cost_a_few_plain_ones(n, hidden, layers):
  # the fp32 matrix instructions take 2.7 times the time of the six bf16 ones
  params, v0 = ml._case(n, hidden, layers, seed=3)
  plan = ml._model(n, params, hidden, layers)[0].plan(ml._dev())
  plain = tuple(torch.as_tensor(x.data, device=ml._dev()) for x in v0)
  huge = tuple(x / x.abs().max() * 3e38 for x in plain)

  def best(fields):
    times = []
    for _ in range(5):
      start, end = torch.cuda.Event(True), torch.cuda.Event(True)
      start.record()
      for _ in range(10):
        plan.tower(*fields)
      end.record()
      end.synchronize()
      times.append(start.elapsed_time(end))
    return min(times)

  assert best(huge) <= 6 * best(plain)


def test_explicit_row_blocks_agree():
  # 9 x 128^2 takes four rows and both components per workgroup, 128^2 one of each
  n, batch = 128, 9
  params, v0 = ml._case(n, 16, 1, seed=5)
  step = ml._model(n, params, 16, 1)[0]
  u, v = (torch.as_tensor(x.data, device=ml._dev()).repeat(batch, 1, 1) for x in v0)
  u[3] *= 0.5
  many, one = step.plan(ml._dev(), batch).step(u, v, 1), step.plan(ml._dev())
  for b in (0, 3, 8):
    for got, want in zip(many, one.step(u[b], v[b], 1)):
      assert torch.equal(got[b], want)
