"""The fitted functions of csrc/nta_torus.h, evaluated in FP32 with fused
multiply-adds from the coefficients in the source (no GPU)."""
import os
import re

import numpy as np
import pytest

F = np.float32
PI = F(3.14159265358979)


def _coefs(name, n):
  src = open(os.path.join(os.path.dirname(__file__), '..',
                          'neural_tangents_amd', 'csrc', 'nta_torus.h')).read()
  body = src[src.index(name):]
  found = [F(x) for x in re.findall(r'(-?\d\.\d+e[-+]\d+)f', body)]
  return found[:n], found[n:]


def _fma(a, b, c):
  return (np.float64(a) * np.float64(b) + np.float64(c)).astype(F)


def _horner(coef, x):
  p = np.full_like(x, coef[0])
  for c in coef[1:]:
    p = _fma(p, x, c)
  return p


def _acos(deg):
  nine, rest = _coefs('float acos_over_sin(', 10)
  return nine if deg == 9 else rest[:8]


def _angle(deg, a):
  """pi - theta as torus_act forms it, for rho = a >= 0."""
  sn = np.sqrt(1.0 - a.astype(np.float64) ** 2).astype(F)
  h = _fma(-sn, _horner(_acos(deg), a), F(0.5) * PI)
  return (F(0.5) * PI + h).astype(F).astype(np.float64)


@pytest.mark.parametrize('deg,bound', [(7, 6.5e-7), (9, 3e-7)])
def test_angle_bound(deg, bound):
  """3.8e-7 and 8e-9 of fit, and the rounding of pi - theta in [2, 4)."""
  a = np.linspace(0.0, 1.0, 400001).astype(F)
  want = np.float64(PI) - np.arccos(a.astype(np.float64))
  got = _angle(deg, a)
  assert np.abs(got - want).max() <= bound
  assert got[-1] == np.float64(PI)
  if deg == 9:
    assert got[0] == np.float64(F(0.5) * PI)


def test_mean_angle_over_intervals():
  """Layers repeat the mean error over the correlations they meet: within
  1.5e-8 on every interval, 5e-8 next to correlation 0 (there the FP32 pi / 2
  itself is 4.4e-8 off); each mean of 40,000 roundings of up to 1.2e-7 is known
  to 1e-9."""
  rng = np.random.default_rng(0)
  edges = [0.0, 0.1, 0.3, 0.5, 0.7, 0.8, 0.87, 0.92, 0.95, 0.97, 0.985, 0.995,
           0.999, 1.0]
  for lo, hi in zip(edges, edges[1:]):
    a = rng.uniform(lo, hi, 40000).astype(F)
    err = _angle(9, a) - (np.float64(PI) - np.arccos(a.astype(np.float64)))
    assert abs(err.mean()) <= (5e-8 if lo < 0.3 else 1.5e-8), (lo, err.mean())


def test_arctangent_bound():
  """atan2_right: 1.5e-8 of fit relative, FP32 rounding of t, z and the
  product, and the hardware reciprocal's 1 ulp (here the rounded quotient)."""
  coef, _ = _coefs('float atan2_right(', 9)
  t = np.geomspace(1e-6, 1.0, 200001).astype(F)
  z = (t * t).astype(F)
  p = _horner(coef, z)
  want = np.arctan(t.astype(np.float64))
  small = (p * t).astype(F)
  assert np.abs(small / want - 1.0).max() <= 2e-7
  big = _fma(-p, t, F(0.5) * PI).astype(np.float64)   # atan(1 / t)
  assert np.abs(big / (0.5 * np.pi - want) - 1.0).max() <= 2e-7
