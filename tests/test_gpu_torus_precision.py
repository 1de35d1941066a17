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
