"""CPU check of the limiter's quotient (fvm.hip ratio): with r0 near 1/d,
r = RN(r0 + RN(1 - d r0) r0), q = RN(x r), RN(q + RN(x - q d) r) is x / d for
|x| <= d, evaluated with exact fused steps for every significand of d and r0
the rounded reciprocal or one of its neighbours.

The claim under test: every quotient is the IEEE one but for the divisor of 24
one bits from an estimate beside the rounded one, where it is one ulp off
(v_rcp_f32 rounds that reciprocal correctly); r itself is the rounded reciprocal for all
but 33 (divisor, estimate) pairs."""
import ctypes
import ctypes.util

import numpy as np

_libm = ctypes.CDLL(ctypes.util.find_library('m') or 'libm.so.6')
_libm.fmaf.restype = ctypes.c_float
_libm.fmaf.argtypes = (ctypes.c_float, ctypes.c_float, ctypes.c_float)
F = np.float32


def _fma(a, b, c):
  """RN(a b + c): the 64-bit sum rounds like the exact one unless it lies
  between two floats; those few go through the C library."""
  s = a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)
  f = s.astype(F)
  tie = np.abs(s - f) >= 0.49 * np.spacing(np.abs(f)).astype(np.float64)
  for i in np.flatnonzero(tie):
    f[i] = _libm.fmaf(a[i], b[i], c[i])
  return f


def _quotient(x, d, r):
  q = x * r
  return _fma(_fma(-q, d, x), r, q)


def test_every_divisor_significand():
  rng = np.random.default_rng(3)
  off_reciprocals, wrong = [], []
  for k in range(32):
    m = np.arange(k << 18, (k + 1) << 18, dtype=np.uint32)
    d = (m | np.uint32(0x3f800000)).view(F)
    rounded = F(1) / d
    xs = [np.ones_like(d), rng.uniform(0.5, 1, d.size).astype(F)]
    for r0 in (np.nextafter(rounded, F(0)), rounded, np.nextafter(rounded, F(4))):
      r = _fma(_fma(-d, r0, np.ones_like(d)), r0, r0)
      off_reciprocals += list(zip(d[r != rounded], r0[r != rounded]))
      for x in xs:
        bad = _quotient(x, d, r) != x / d
        wrong += list(zip(x[bad], d[bad], r0[bad]))
  ones = F(2 - 2.0 ** -23)
  assert all(d == ones and r0 != F(1) / ones for _, d, r0 in wrong), wrong[:4]
  assert len(off_reciprocals) == 33
  # the pairs whose reciprocal is off, with many dividends
  for d, r0 in off_reciprocals:
    if d == ones:
      continue
    x = (rng.uniform(0, 1, 1 << 16) * d).astype(F)
    dd, rr = np.full_like(x, d), np.full_like(x, r0)
    r = _fma(_fma(-dd, rr, np.ones_like(x)), rr, rr)
    assert np.array_equal(_quotient(x, dd, r), x / dd), (d, r0)


def test_divisor_of_ones():
  m = np.arange(1 << 20, dtype=np.uint32) * np.uint32(8) + np.uint32(7)
  x = np.concatenate([(m | np.uint32(0x3f000000)).view(F), (m | np.uint32(0x3f800000)).view(F), [F(1)]])
  d = np.full_like(x, F(2 - 2.0 ** -23))
  r = np.full_like(x, F(1) / d[0])  # what v_rcp_f32 gives, and what a step from it keeps
  assert _fma(_fma(-d[:1], r[:1], np.ones(1, F)), r[:1], r[:1])[0] == r[0]
  assert np.array_equal(_quotient(x, d, r), x / d)


def test_ranges_ends():
  # the smallest and largest divisors, and dividends down to 2^-100
  rng = np.random.default_rng(4)
  for e in (-126, -100, 0, 100, 125):
    d = (rng.uniform(1, 2, 1 << 16) * 2.0 ** e).astype(F)
    x = (d * 2.0 ** -rng.uniform(0, min(60, e + 100) if e > -100 else 0, d.size)).astype(F)
    x = np.minimum(x, d)
    r0 = F(1) / d
    r = _fma(_fma(-d, r0, np.ones_like(d)), r0, r0)
    got, want = _quotient(x, d, r), x / d
    exact = np.abs(x) >= F(2.0 ** -100)
    assert np.array_equal(got[exact], want[exact]), e
    assert (np.abs(got.astype(np.float64) - want) <= np.spacing(want)).all(), e
  # 2^126 itself, whose reciprocal is the smallest normal number
  d = np.full(1 << 12, F(2.0 ** 126))
  x = (rng.uniform(0, 1, d.size) * 2.0 ** 126).astype(F)
  assert np.array_equal(_quotient(x, d, F(1) / d), x / d)
