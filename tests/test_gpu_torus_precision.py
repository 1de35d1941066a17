"""Deep networks on the register-resident kernels against the FP64 oracle:
errors of the maps that every layer repeats would add up (needs a GPU)."""
import numpy as np
import pytest

from conftest import rel_err
from neural_tangents_amd import stax
from neural_tangents_amd.data import blurred_images
from oracle import stax_oracle as so

pytestmark = pytest.mark.gpu


def _layers(depth, readout):
  net = [stax.Conv(1, (3, 3), padding='SAME', W_std=2.0 ** 0.5),
         stax.Relu()] * depth
  ref = [so.conv_layer(W_std=2.0 ** 0.5, b_std=0.0), so.relu_layer()] * depth
  if readout == 'flat':
    net += [stax.Flatten()]
    ref += [so.flatten_layer()]
  else:
    net += [stax.GlobalAvgPool()]
    ref += [so.global_avg_pool_layer()]
  return (stax.serial(*net, stax.Dense(1))[2], ref + [so.dense_layer()])


@pytest.mark.parametrize('side', [8, 13, 16])
@pytest.mark.parametrize('readout', ['flat', 'gap'])
def test_21_layers(side, readout):
  """The mean error of pi - theta (1.1e-8 of at least pi / 2, over most layers
  of about 3) adds up to 8e-8 of the ntk at most over 21 layers; the outputs'
  own rounding is 3e-8."""
  x1, x2 = blurred_images([3, 4], side, seed=side)
  kfn, ref = _layers(21, readout)
  k = kfn(x1, x2, ('nngp', 'ntk'))
  want = so.kernel_fn(ref, x1.astype(np.float64), x2.astype(np.float64),
                      ('nngp', 'ntk'))
  for f in ('nngp', 'ntk'):
    e = rel_err(getattr(k, f).double().cpu().numpy(), want[f])
    assert e <= 1e-7, (f, e)


@pytest.mark.parametrize('side,depths,tol', [
    (16, (21,), 1e-6), (16, (3, 3, 3), 1e-6), (32, (10,), 1e-6),
    (32, (2, 1, 1), 3e-6), (32, (3, 3, 3), 3e-6)])
def test_copies_of_images(side, depths, tol):
  """An image against its copy: 1e-6, FP32 rounding, where the map is exact up
  to correlation 1.  The 32x32 segment before a pool rounds the correlation
  (three roundings, so the angle by up to 6e-4 and pi - theta by 1.9e-4 of
  itself) on the spatial diagonal, 1 / 1024 of the elements, which weigh up to
  five times the mean, in each of up to three layers."""
  net, ref = [], []
  for k in depths:
    net += [stax.Conv(1, (3, 3), padding='SAME', W_std=2.0 ** 0.5),
            stax.Relu()] * k
    ref += [so.conv_layer(W_std=2.0 ** 0.5, b_std=0.0), so.relu_layer()] * k
    if len(depths) > 1:
      net.append(stax.AvgPool((2, 2), (2, 2)))
      ref.append(so.avg_pool_layer((2, 2), (2, 2)))
  kfn = stax.serial(*net, stax.GlobalAvgPool(), stax.Dense(1))[2]
  ref += [so.global_avg_pool_layer(), so.dense_layer()]
  x = blurred_images([24], side, channels=1, seed=4)[0]
  k = kfn(x, x.copy(), ('nngp', 'ntk'))
  for i in (0, 11, 23):
    want = so.kernel_fn(ref, x[i:i + 1].astype(np.float64), None,
                        ('nngp', 'ntk'))
    for f in ('nngp', 'ntk'):
      w = float(want[f][0, 0])
      assert abs(float(getattr(k, f)[i, i]) - w) <= tol * abs(w), (i, f)
