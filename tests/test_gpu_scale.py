"""Kernels of networks without biases are homogeneous: inputs times s give
s^2 K, and W_std of all L convolutions times s gives s^(2 L) K, bit for bit
where s is a power of two and no product leaves FP32's normal range (needs a
GPU).  The exact ReLU map squares normalisers, so this is what it owes small
and large ones (small W_std through many layers, images that are not
normalised)."""
import pytest
import torch

from neural_tangents_amd import _engine, grad, stax
from neural_tangents_amd.data import blurred_images

pytestmark = pytest.mark.gpu


def _net(kind, W):
  def layers(n):
    return [stax.Conv(1, (3, 3), padding='SAME', W_std=W), stax.Relu()] * n
  pool = [stax.AvgPool((2, 2), (2, 2))]
  if kind == 'flat':
    return stax.serial(*layers(12), stax.Flatten(), stax.Dense(1))[2], 12
  if kind == 'gap':
    return stax.serial(*layers(12), stax.GlobalAvgPool(),
                       stax.Dense(1))[2], 12
  return stax.serial(*layers(3), *pool, *layers(3), *pool, *layers(2),
                     stax.GlobalAvgPool(), stax.Dense(1))[2], 8


def _images(side, C=3):
  return [torch.from_numpy(x).cuda()
          for x in blurred_images([3, 4], side, channels=C, seed=side)]


@pytest.mark.parametrize('side', [8, 12, 16, 20, 32])
@pytest.mark.parametrize('kind', ['myrtle', 'gap', 'flat'])
@pytest.mark.parametrize('what,s', [
    ('x', 2.0 ** -30), ('x', 2.0 ** 30), ('W', 2.0 ** -2), ('W', 2.0 ** -4),
    ('W', 2.0 ** 3)])
def test_convolutional_networks(kind, side, what, s):
  x1, x2 = _images(side)
  W = 2.0 ** 0.5
  kfn, L = _net(kind, W)
  if what == 'W':
    scaled, fac = _net(kind, W * s)[0], s ** (2 * L)
    got = [scaled(x1, x, ('nngp', 'ntk')) for x in (x2, None)]
  else:
    fac = s * s
    got = [kfn(x1 * s, None if x is None else x * s, ('nngp', 'ntk'))
           for x in (x2, None)]
  for k, x in zip(got, (x2, None)):
    want = kfn(x1, x, ('nngp', 'ntk'))
    for f in ('nngp', 'ntk'):
      w = getattr(want, f).double()
      assert torch.equal(getattr(k, f).double() / fac, w), f


@pytest.mark.parametrize('side', [8, 12])
def test_self_covariance(side):
  x1, _ = _images(side)
  kfn, _ = _net('flat', 2.0 ** 0.5)
  want = kfn(x1)
  got = kfn(x1 * 2.0 ** -30)
  assert torch.equal(got.cov1.double() * 2.0 ** 60, want.cov1.double())


@pytest.mark.parametrize('side', [8, 16, 32])
@pytest.mark.parametrize('same', [True, False])
@pytest.mark.parametrize('b', [0.0, 0.1])
def test_gradients(side, same, b):
  """Images and b_std times s: K times s^2, its gradients in them times s, in
  W_std times s^2."""
  xs = _images(side)
  s = 2.0 ** -30

  def run(scale):
    xa, xb = (x.mul(scale).requires_grad_() for x in xs)
    W = torch.tensor(2.0 ** 0.5, device='cuda', requires_grad=True)
    bs = torch.tensor(b * scale, device='cuda', requires_grad=True)
    n, t = grad.kernel(xa, None if same else xb, W, bs,
                       grad.myrtle_builder((2, 1, 1)))
    return torch.autograd.grad((n + t).sum(),
                               [W, bs, xa] + ([] if same else [xb]))
  want, got = run(1.0), run(s)
  for g, w in zip(got[2:], want[2:]):
    assert torch.equal(g.double() / s, w.double())
  # FP64 sums of FP32 products
  for g, w, fac in ((got[0], want[0], s * s), (got[1], want[1], s)):
    assert abs(float(g) / fac - float(w)) <= 1e-6 * abs(float(w))


@pytest.mark.parametrize('n1,n2', [(5, 9), (90, 0), (1500, 1400)])
def test_fully_connected(n1, n2):
  """Rows whose normalisers' products are subnormal, or large: 1e-5, the bar of
  the other kernel tests (two evaluations of one map; the subnormal product,
  2^-128, is resolved to 5e-7)."""
  g = torch.Generator(device='cuda').manual_seed(n1)
  x1 = torch.randn((n1, 20), generator=g, device='cuda')
  x2 = torch.randn((n2, 20), generator=g, device='cuda') if n2 else None
  net = [stax.Dense(1, 2.0 ** 0.5), stax.Relu()] * 6 + [stax.Dense(1)]
  kfn = stax.serial(*net)[2]
  assert _engine._is_flat(kfn.plan(x1.shape), (n1, 1, 1, 20))
  want = kfn(x1, x2, ('nngp', 'ntk'))
  for s in (2.0 ** -32, 2.0 ** 28):
    got = kfn(x1 * s, None if x2 is None else x2 * s, ('nngp', 'ntk'))
    for f in ('nngp', 'ntk'):
      w = getattr(want, f).double()
      d = getattr(got, f).double() / s ** 2 - w
      assert d.norm() <= 1e-5 * w.norm(), f
