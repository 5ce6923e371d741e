"""Launch shapes picked from a launch's size: each must step bit-identically to
the same plan with one-row, one-column tiles set by hand (tile shapes never
change results), on both sides of every line of the rules (where the shapes have
to differ, so a line that moves is noticed), for whole batches and for short slot
lists of a large batch."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev():
  return torch.device('cuda', 0)


def _fvm(n, batch, **kw):
  import dataclasses
  from jax_cfd_amd import serving
  from jax_cfd_amd.base import _fvm
  spec = dataclasses.replace(serving.FvmFamily(n, _dev()).spec, **kw)
  gen = torch.Generator(device=_dev()).manual_seed(n + batch)
  u = torch.randn((batch, n, n), device=_dev(), generator=gen)
  v = torch.randn((batch, n, n), device=_dev(), generator=gen)
  return _fvm.FvmPlan(spec, _dev(), batch=batch), u, v


@pytest.mark.parametrize("n,batch", [(32, 7), (32, 32), (32, 512), (64, 7), (64, 8), (64, 15), (64, 64),
                                     (64, 256), (128, 7), (128, 8), (128, 31), (128, 128),
                                     (256, 2), (256, 3), (256, 4), (256, 16), (256, 47), (256, 48),
                                     (512, 2), (512, 8), (512, 15), (512, 16), (1024, 1), (1024, 3)])
def test_fvm_rule_steps_as_one_row_tiles(n, batch):
  plan, u, v = _fvm(n, batch)
  if batch == 1:
    u, v = u[0], v[0]
  got = plan.step(u, v, 2)
  plan.set_tiles(1, 1, 1, 8)
  want = plan.step(u, v, 2)
  print(f"n={n} batch={batch}", flush=True)
  assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("n,batch", [(32, 64), (128, 40), (256, 48), (512, 16)])
def test_fvm_short_slot_lists(n, batch):
  plan, u, v = _fvm(n, batch)
  want = plan.step(u, v, 2)
  slots = torch.tensor([batch - 1, 0, 2], dtype=torch.int32, device=_dev())
  u1, v1 = u.clone(), v.clone()
  plan.step_slots(u1, v1, slots, 2)
  idx = slots.long()
  assert torch.equal(u1[idx], want[0][idx]) and torch.equal(v1[idx], want[1][idx])
  assert torch.equal(u1[1], u[1])


# row kernels without a tunable shape: one row per workgroup for few rows
@pytest.mark.parametrize("kw", [dict(diffusion=1), dict(rk_stages=2, rk_a=(1.0,), rk_b=(0.5, 0.5))])
@pytest.mark.parametrize("n,batch", [(32, 33), (128, 9), (256, 4), (512, 2)])
def test_fvm_untuned_kernels_match_lone_instances(n, batch, kw):
  plan, u, v = _fvm(n, batch, **kw)
  one, _, _ = _fvm(n, 1, **kw)
  got = plan.step(u, v, 2)
  for k in (0, batch - 1):
    want = one.step(u[k].contiguous(), v[k].contiguous(), 2)
    assert torch.equal(got[0][k], want[0]) and torch.equal(got[1][k], want[1])


@pytest.mark.parametrize("n,batch", [(32, 63), (32, 64), (64, 16), (64, 32), (64, 256), (128, 7),
                                     (128, 8), (128, 64), (256, 15), (256, 16), (512, 1),
                                     (512, 31), (512, 32), (1024, 2), (1024, 16)])
def test_spectral_rule_steps_as_one_column_tiles(n, batch):
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  plan = _ns2d.Ns2dPlan(serving.SpectralFamily(n, _dev()).spec, batch, _dev())
  gen = torch.Generator(device=_dev()).manual_seed(n + batch)
  w = plan.rfft2(torch.randn((batch, n, n), device=_dev(), generator=gen))
  got = plan.step(w, 2)
  plan.set_tiles(1, 1, 8)
  assert torch.equal(got, plan.step(w, 2))
  if batch > 3:
    slots = torch.tensor([batch - 1, 1], dtype=torch.int32, device=_dev())
    other = _ns2d.Ns2dPlan(plan.spec, batch, _dev())
    w1 = w.clone()
    other.step_slots(w1, slots, 2)
    assert torch.equal(w1[slots.long()], got[slots.long()])


# batches above 2^23 cells run in parts: even and uneven splits, with and
# without a slot list
@pytest.mark.parametrize("n,batch", [(256, 128), (256, 129), (512, 33)])
def test_spectral_batches_in_parts_match_lone_instances(n, batch):
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  spec = serving.SpectralFamily(n, _dev()).spec
  plan, one = _ns2d.Ns2dPlan(spec, batch, _dev()), _ns2d.Ns2dPlan(spec, 1, _dev())
  gen = torch.Generator(device=_dev()).manual_seed(batch)
  w = plan.rfft2(torch.randn((batch, n, n), device=_dev(), generator=gen))
  got = plan.step(w, 34)  # one direct step, one 32-step graph, one direct step
  perm = torch.randperm(batch, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(_dev())
  ws = w.clone()
  plan.step_slots(ws, perm, 34)
  assert torch.equal(ws, got)
  for k in (0, batch // 2 - 1, batch // 2, batch - 1):
    assert torch.equal(got[k], one.step(w[k].contiguous(), 34)), k


# an output that overlaps the input: nothing is written before all is read
@pytest.mark.parametrize("batch,shift", [(9, 1), (9, -1), (17, 4)])
def test_spectral_parts_with_overlapping_output(batch, shift):
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  n = 1024
  plan = _ns2d.Ns2dPlan(serving.SpectralFamily(n, _dev()).spec, batch, _dev())
  gen = torch.Generator(device=_dev()).manual_seed(batch)
  w = plan.rfft2(torch.randn((batch, n, n), device=_dev(), generator=gen))
  want = plan.step(w, 2)
  both = torch.zeros((batch + abs(shift), n, n // 2 + 1), dtype=torch.complex64, device=_dev())
  first, second = both[:batch], both[abs(shift):]
  src, dst = (first, second) if shift > 0 else (second, first)
  src.copy_(w)
  plan.step(src, 2, out=dst)
  assert torch.equal(dst, want)
  same = w.clone()
  plan.step(same, 2, out=same)
  assert torch.equal(same, want)


# more parts than have graphs of their own
def test_spectral_batch_in_many_parts():
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  n, batch = 1024, 137
  spec = serving.SpectralFamily(n, _dev()).spec
  plan, one = _ns2d.Ns2dPlan(spec, batch, _dev()), _ns2d.Ns2dPlan(spec, 1, _dev())
  gen = torch.Generator(device=_dev()).manual_seed(batch)
  w = one.rfft2(torch.randn((n, n), device=_dev(), generator=gen))
  ws = w[None] * torch.linspace(0.5, 1.5, batch, device=_dev())[:, None, None]
  got = plan.step(ws, 33)
  for k in (0, 60, 136):
    assert torch.equal(got[k], one.step(ws[k].contiguous(), 33)), k


# every wavefront layout of the column and row kernels, on instances whose
# forcing list is longer than the registers hold and reaches column n / 2
@pytest.mark.parametrize("n", [32, 64, 128, 256, 512, 1024])
def test_spectral_tiles_with_long_forcing_lists(n):
  import dataclasses
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  spec = dataclasses.replace(
      serving.SpectralFamily(n, _dev()).spec,
      forcing=tuple((p % n, c, 3.0 + p, -1.5 * c) for p, c in
                    ((0, 4), (n - 4, 0), (n // 2, n // 2), (3, n // 2), (n - 1, n // 2 - 1), (5, 7))))
  plan = _ns2d.Ns2dPlan(spec, 2, _dev())
  gen = torch.Generator(device=_dev()).manual_seed(n)
  w = plan.rfft2(torch.randn((2, n, n), device=_dev(), generator=gen))
  plan.set_tiles(1, 1, 8)
  want = plan.step(w, 2)
  for cols, rows in ((2, 2), (4, 4), (8, 8), (16, 16), (8, 2), (16, 4), (2, 8), (4, 2)):
    try:
      plan.set_tiles(cols, rows, 8)
    except NotImplementedError:
      continue
    print(f"n={n} cols={cols} rows={rows}", flush=True)
    assert torch.equal(plan.step(w, 2), want), (cols, rows)
  # the forcing list itself: the explicit terms of a zero state are the list
  f = plan.explicit_terms(torch.zeros_like(w))
  for p, c, re, im in spec.forcing:
    assert f[1, p, c].item() == complex(re, im)


# rows of 1024 march with a thread per cell: every tile, scheme and batch
# against one-row tiles, which stage their rows
@pytest.mark.parametrize("convect", [0, 1, 2, 3])
@pytest.mark.parametrize("batch", [1, 2])
def test_fvm_marching_rows_of_1024(convect, batch):
  plan, u, v = _fvm(1024, batch, convect=convect)
  if batch == 1:
    u, v = u[0], v[0]
  plan.set_tiles(1, 1, 1, 8)
  want = plan.step(u, v, 2)
  for rows in (4, 8, 16, 32):
    plan.set_tiles(rows, 1, 1, 8)
    got = plan.step(u, v, 2)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), rows


# kernel times are those of the launches a step makes: with parts, their sum
# over a step is the step's own time but for launch gaps (one launch over all of
# 64 x 512^2, beyond the cache, adds up to 1.2 steps)
@pytest.mark.parametrize("n,batch", [(512, 64), (256, 256)])
def test_spectral_kernel_times_add_up(n, batch):
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  plan = _ns2d.Ns2dPlan(serving.SpectralFamily(n, _dev()).spec, batch, _dev())
  w = 0.01 * plan.rfft2(torch.randn((batch, n, n), device=_dev(),
                                    generator=torch.Generator(device=_dev()).manual_seed(n)))
  plan.set_graphs(False)  # direct launches, as the kernel times are
  times = []
  for _ in range(5):
    start, end = torch.cuda.Event(True), torch.cuda.Event(True)
    start.record()
    plan.step(w, 33, out=w)
    end.record()
    end.synchronize()
    times.append(start.elapsed_time(end) / 33)
  ms = plan.time_kernels(w, 20)
  total = sum(ms[k] * plan.LAUNCHES_PER_STEP[k] for k in ms)
  print(f"{batch} x {n}^2: step {min(times):.3f} ms, kernels {total:.3f} ms", flush=True)
  assert 0.8 * min(times) <= total <= 1.1 * min(times)


# (n, rows over all instances from which a rule picks another shape)
FVM_LINES = [(n, rows) for n, lines in {
    32: (1024, 2048, 4096, 16384), 64: (1024, 2048, 4096, 16384), 128: (1024, 2048, 4096, 16384, 32768),
    256: (1024, 2048, 4096, 8192), 512: (1024, 2048, 4096), 1024: (2048, 4096, 16384)}.items() for rows in lines]
SPECTRAL_LINES = [(n, rows) for n, lines in {
    32: (2048, 8192), 64: (2048, 16384), 128: (1024, 2048, 4096, 8192, 16384), 256: (512, 1024, 4096, 8192),
    512: (4096,), 1024: (2048, 4096)}.items() for rows in lines]


@pytest.mark.parametrize("n,rows", FVM_LINES)
def test_fvm_rules_on_both_sides(n, rows):
  below, above = _fvm(n, rows // n - 1), _fvm(n, rows // n)
  assert below[0].tiles != above[0].tiles
  for plan, u, v in (below, above):
    u, v = u.reshape(plan.shape), v.reshape(plan.shape)
    got = plan.step(u, v, 2)
    plan.set_tiles(1, 1, 1, 8)
    want = plan.step(u, v, 2)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("n,rows", SPECTRAL_LINES)
def test_spectral_rules_on_both_sides(n, rows):
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  spec = serving.SpectralFamily(n, _dev()).spec
  plans = [_ns2d.Ns2dPlan(spec, rows // n - k, _dev()) for k in (1, 0)]
  assert plans[0].tiles != plans[1].tiles
  for plan in plans:
    gen = torch.Generator(device=_dev()).manual_seed(n + plan.batch)
    w = plan.rfft2(torch.randn(plan.real_shape, device=_dev(), generator=gen))
    got = plan.step(w, 2)
    plan.set_tiles(1, 1, 8)
    assert torch.equal(got, plan.step(w, 2))


# the marching stencil at its other sizes, and a group's, whose workgroups hold
# two cells of a 512 row per thread: every scheme against one-row tiles
@pytest.mark.parametrize("convect", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [256, 512])
def test_fvm_marching_rows_of_every_scheme(n, convect):
  from jax_cfd_amd.base import _fvm as fvm
  plan, u, v = _fvm(n, 2, convect=convect)
  plan.set_tiles(1, 1, 1, 8)
  want = plan.step(u, v, 2)
  for rows in (16, 32):
    plan.set_tiles(rows, 1, 1, 8)
    got = plan.step(u, v, 2)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), rows
  gu, gv = u.clone(), v.clone()
  fvm.FvmGroup(_dev()).step([(plan, gu, gv, [0, 1])], 2)
  assert torch.equal(gu, want[0]) and torch.equal(gv, want[1])


# wavenumbers of other boxes: the register kernels form them from the box's
# length, the staged ones read the table
@pytest.mark.parametrize("n,batch", [(32, 256), (64, 256), (128, 128), (256, 64), (512, 16), (1024, 4)])
@pytest.mark.parametrize("box", [(1.0, 3.0), (10.7, 0.3), (3.141592653589793, 100.0)])
def test_spectral_boxes_step_as_one_column_tiles(n, batch, box):
  import dataclasses
  from jax_cfd_amd import serving
  from jax_cfd_amd.spectral import _ns2d
  spec = dataclasses.replace(serving.SpectralFamily(n, _dev()).spec, dx=box[0] / n, dy=box[1] / n, dt=1e-5)
  plan = _ns2d.Ns2dPlan(spec, batch, _dev())
  gen = torch.Generator(device=_dev()).manual_seed(n)
  w = 0.01 * plan.rfft2(torch.randn((batch, n, n), device=_dev(), generator=gen))
  got = plan.step(w, 2)
  plan.set_tiles(1, 1, 8)
  assert torch.isfinite(torch.view_as_real(got)).all() and torch.equal(got, plan.step(w, 2))
