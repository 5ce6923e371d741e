"""The jcfd_tensor that a tensor is passed as, against its DLPack structure."""
import ctypes

import pytest
import torch
import torch.utils.dlpack

from jax_cfd_amd import _lib


class _Tensor(ctypes.Structure):
  _fields_ = [('data', ctypes.c_void_p), ('device_type', ctypes.c_int32), ('device_id', ctypes.c_int32),
              ('ndim', ctypes.c_int32), ('code', ctypes.c_uint8), ('bits', ctypes.c_uint8),
              ('lanes', ctypes.c_uint16), ('shape', ctypes.POINTER(ctypes.c_int64)),
              ('strides', ctypes.POINTER(ctypes.c_int64)), ('byte_offset', ctypes.c_uint64)]


def _fields(address):
  t = _Tensor.from_address(address)
  shape = list(t.shape[:t.ndim])
  strides, step = [], 1
  for k in reversed(range(t.ndim)):
    strides.insert(0, t.strides[k] if t.strides else step)
    step *= shape[k]
  return ((t.data or 0) + t.byte_offset, t.device_type, t.device_id, t.code, t.bits, t.lanes, shape, strides)


def _dlpack(t):
  cap = torch.utils.dlpack.to_dlpack(t)
  return _fields(_lib._PyCapsule_GetPointer(cap, b'dltensor'))


@pytest.mark.gpu
def test_arguments_cost_no_more_than_their_capsules():
  # the capsules and pointers themselves, with the loop around them
  import timeit
  ts = [torch.zeros(32, 32, device='cuda') for _ in range(4)]

  def args():
    with _lib.dlpack_args() as dl:
      for t in ts:
        dl(t)

  def capsules():
    caps = []
    for t in ts:
      caps.append(torch.utils.dlpack.to_dlpack(t))
      _lib._PyCapsule_GetPointer(caps[-1], b'dltensor')

  best = [min(timeit.repeat(f, number=2000, repeat=7)) for f in (args, capsules)]
  assert best[0] <= 2 * best[1]


def test_other_tensors_go_as_dlpack():
  with _lib.dlpack_args() as dl:
    for t in (torch.zeros(8, 8), torch.zeros(8, 8).T, torch.zeros(1, 8, 8), torch.zeros(8, dtype=torch.float64)):
      assert _fields(dl(t)) == _dlpack(t)


@pytest.mark.gpu
def test_gpu_tensors():
  x = torch.zeros(4, 32, 32, device='cuda')
  c = torch.zeros(32, 17, dtype=torch.complex64, device='cuda')
  with _lib.dlpack_args() as dl:
    for t in (x, x[1], x[1:3], x[:1], x[:, :, 1], x.transpose(1, 2), c, c.conj(), c.real,
              torch.zeros(4, dtype=torch.int32, device='cuda'), x.double()):
      assert _fields(dl(t)) == _dlpack(t)
