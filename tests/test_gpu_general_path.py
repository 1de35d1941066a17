"""The general path's fused launches on networks with a readout, which the
register-resident segments take by themselves: forced onto the general path,
with the entry points that ran (needs a GPU).  Against the same network stage
by stage (both FP32: 1e-5 relative, 1e-4 of the largest entry elementwise) and
the FP64 oracle (1e-5)."""
import numpy as np
import pytest
import torch

from conftest import rel_err
from neural_tangents_amd import _engine, stax
from neural_tangents_amd.data import blurred_images
from oracle import stax_oracle as so

pytestmark = pytest.mark.gpu

FUSED = {2: 'nta_first_pool_stage', 3: 'nta_first3_pool_stage'}


@pytest.fixture
def general(monkeypatch):
  monkeypatch.setattr(_engine, '_torus_segments', lambda plan, shape: None)
  return monkeypatch


def _net(fused):
  layers = []
  for w in (1.3, 1.5, 1.2)[:fused]:
    layers += [stax.Conv(1, (3, 3), padding='SAME', W_std=w), stax.Relu()]
  layers += [stax.AvgPool((2, 2), (2, 2)),
             stax.Conv(1, (3, 3), padding='SAME', W_std=1.4), stax.Relu(),
             stax.AvgPool((2, 2), (2, 2)), stax.GlobalAvgPool(),
             stax.Dense(1, 1.0, 0.0)]
  return stax.serial(*layers)[2]


def _traced(m, *a, **kw):
  """The call's result and the entry points it launched, in order."""
  m.setattr(_engine, 'TRACE', [])
  k = a[0](*a[1:], **kw)
  names = [t[0].split('[')[0] for t in _engine.TRACE]
  m.setattr(_engine, 'TRACE', None)
  assert not any(n.startswith('nta_torus') for n in names)
  return k, names


def _close(a, b, name):
  a, b = (v.double().cpu().numpy() for v in (a, b))
  e = np.linalg.norm(a - b) / np.linalg.norm(b)
  assert e <= 1e-5, (name, e)
  assert np.max(np.abs(a - b)) <= 1e-4 * np.max(np.abs(b)), name


@pytest.mark.parametrize('fused', [2, 3])
@pytest.mark.parametrize('same', [True, False])
@pytest.mark.parametrize('tiled', [False, True])
def test_fused_matches_stagewise(general, fused, same, tiled):
  x1, x2 = blurred_images([5, 3], 32, seed=fused)
  x2 = None if same else x2
  kfn = _net(fused)
  # tiles of four pairs' pooled states: several launches a matrix, symmetric
  # ones for x2 = None
  kw = {'tile_bytes': 4 * 2 * 2 * 4 * 16 ** 4} if tiled else {}
  f, names = _traced(general, kfn, x1, x2, ('nngp', 'ntk'), **kw)
  assert names.count(FUSED[fused]) == (1 if not tiled else 6 if same else 5)
  assert names.count('nta_qnorm') == fused * (1 if same else 2)
  with general.context() as m:
    m.setattr(_engine, '_fused_stages', lambda plan, shape: 0)
    p, names = _traced(m, kfn, x1, x2, ('nngp', 'ntk'))
  assert 'nta_stage' in names and FUSED[fused] not in names
  _close(f.nngp, p.nngp, 'nngp')
  _close(f.ntk, p.ntk, 'ntk')
  if same:
    assert torch.equal(f.ntk, f.ntk.T)


@pytest.mark.parametrize('depth,fused', [(5, 2), (10, 3)])
def test_fused_matches_oracle(general, depth, fused):
  x1, x2 = blurred_images([2, 3], 32, seed=0)
  k, names = _traced(general, stax.myrtle(depth)[2], x1, x2, ('nngp', 'ntk'))
  assert FUSED[fused] in names
  depths = {5: (2, 1, 1), 10: (3, 3, 3)}[depth]
  ref = so.kernel_fn(so.myrtle_layers(depths), x1, x2, ('nngp', 'ntk'))
  for g in ('nngp', 'ntk'):
    e = rel_err(getattr(k, g).double().cpu().numpy(), ref[g])
    assert e <= 1e-5, (g, e)


def test_segments_take_these_networks():
  """What the other tests of a readout network now run."""
  x1, x2 = blurred_images([2, 3], 32, seed=0)
  for fused in (2, 3):
    kfn = _net(fused)
    assert _engine._torus_segments(kfn.plan(x1.shape), x1.shape) is not None


@pytest.mark.parametrize('fused', [2, 3])
def test_networks_that_stay(monkeypatch, fused):
  """A 5x5 convolution after the pool leaves the fused launches in place."""
  x1, x2 = blurred_images([2, 3], 32, seed=0)
  layers = []
  for w in (1.3, 1.5, 1.2)[:fused]:
    layers += [stax.Conv(1, (3, 3), padding='SAME', W_std=w), stax.Relu()]
  kfn = stax.serial(*layers, stax.AvgPool((2, 2), (2, 2)),
                    stax.Conv(1, (5, 5), padding='SAME'), stax.Relu(),
                    stax.GlobalAvgPool(), stax.Dense(1))[2]
  _, names = _traced(monkeypatch, kfn, x1, x2, ('nngp', 'ntk'))
  assert FUSED[fused] in names
