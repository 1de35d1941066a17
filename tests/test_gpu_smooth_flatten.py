"""Erf and Gelu networks with a Flatten readout, or a global average of small
images, at sizes whose lanes and rows do not fit the wave: elements outside the
images must not reach them (needs a GPU).  Against the general path, 1e-5, the
bar of the other kernel tests."""
import pytest
import torch

from conftest import rel_err
from neural_tangents_amd import _engine, stax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('H,W', [(6, 32), (22, 28), (30, 30), (26, 17),
                                 (5, 19), (13, 13), (9, 7)])
@pytest.mark.parametrize('act', ['erf', 'gelu'])
@pytest.mark.parametrize('head', ['flat', 'gap'])
@pytest.mark.parametrize('scale', [1.0, 60.0])
def test_matches_general_path(monkeypatch, H, W, act, head, scale):
  g = torch.Generator(device='cuda').manual_seed(H * 100 + W)
  n1, n2 = (40, 30) if head == 'flat' else (4, 3)
  x1, x2 = (scale * torch.randn((n, H, W, 1), generator=g, device='cuda')
            for n in (n1, n2))
  layers = []
  for w in (1.3, 1.5, 0.9):
    layers += [stax.Conv(1, (3, 3), padding='SAME', W_std=w),
               stax.Erf(1.1, 0.8, 0.2) if act == 'erf' else stax.Gelu()]
  kfn = stax.serial(*layers, stax.Flatten() if head == 'flat' else
                    stax.GlobalAvgPool(), stax.Dense(1))[2]
  plan = kfn.plan(x1.shape)
  assert (_engine._torus_diag(plan, x1.shape) if head == 'flat' else
          _engine._torus_segments(plan, x1.shape)) is not None
  for x in (x2, None):
    got = kfn(x1, x, ('nngp', 'ntk'))
    with monkeypatch.context() as m:
      m.setattr(_engine, '_torus_diag', lambda plan, shape: None)
      m.setattr(_engine, '_torus_segments', lambda plan, shape: None)
      want = kfn(x1, x, ('nngp', 'ntk'))
    for a, b in zip(got, want):
      a, b = (v.double().cpu().numpy() for v in (a, b))
      assert rel_err(a, b) <= 1e-5
