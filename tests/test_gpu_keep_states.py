"""Pair states kept for the backward are bounded over all live calls, given
back with them and change no result (needs a GPU)."""
import threading

import pytest
import torch

from neural_tangents_amd import _engine, grad
from neural_tangents_amd.data import blurred_images

pytestmark = pytest.mark.gpu

PAIR = 4 * 2 * (16 ** 4 + 8 ** 4)       # bytes of a 32x32 pair's states


def _images(n, seed):
  return torch.from_numpy(blurred_images([n], 32, seed=seed)[0]).cuda()


def _call(x, y):
  a = x.clone().requires_grad_()
  n, t = grad.kernel(a, y, 1.4, 0.1, grad.myrtle_builder((2, 1, 1)))
  return a, (n + t).sum()


def _held():
  torch.cuda.synchronize()
  return torch.cuda.memory_allocated()


def test_live_calls_share_the_bound(monkeypatch):
  """Eight calls of 24 pairs whose graphs live, room for the states of two."""
  x, ys = _images(4, 1), [_images(6, k) for k in range(8)]
  alone = [torch.autograd.grad(loss, a)[0]
           for a, loss in (_call(x, y) for y in ys)]
  need = 24 * PAIR
  monkeypatch.setattr(_engine, 'KEEP_BYTES', 2 * need + need // 2)
  start = _held()
  live = [_call(x, y) for y in ys]
  # images, results and losses are small beside a call's 12 MiB of states
  assert 2 * need <= _held() - start <= 2 * need + 8 * (1 << 20)
  for (a, loss), want in zip(live, alone):
    assert torch.equal(torch.autograd.grad(loss, a)[0], want)
  del live, a, loss
  start = _held()
  again = [_call(x, y) for y in ys[:3]]       # given back: room again
  assert 2 * need <= _held() - start <= 2 * need + 3 * (1 << 20)
  del again


def test_backward_gives_back(monkeypatch):
  """The graph's buffers go with the backward, though the loss is alive."""
  x, y = _images(4, 1), _images(6, 2)
  monkeypatch.setattr(_engine, 'KEEP_BYTES', 24 * PAIR)
  losses = []
  for _ in range(3):
    start = _held()
    a, loss = _call(x, y)
    assert _held() - start >= 24 * PAIR
    loss.backward()
    losses.append((a, loss))


def test_nothing_is_kept_without_gradients(monkeypatch):
  asked = []
  monkeypatch.setattr(_engine, '_kept_states',
                      lambda *a: asked.append(a))
  x, y = _images(3, 1), _images(2, 2)
  with torch.no_grad():
    grad.kernel(x.requires_grad_(), y, 1.4, 0.1, grad.myrtle_builder())
  assert not asked


def test_function_with_five_arguments():
  x, y = _images(3, 1), _images(2, 2)
  a, loss = _call(x, y)
  want = torch.autograd.grad(loss, a)[0]
  b = x.clone().requires_grad_()
  n, t = grad.KernelFunction.apply(b, y, 1.4, 0.1,
                                   grad.myrtle_builder((2, 1, 1)))
  assert torch.equal(torch.autograd.grad((n + t).sum(), b)[0], want)


def test_threads():
  """Calls of several threads and streams count once each."""
  x, ys = _images(3, 1), [_images(4, k) for k in range(4)]
  want = [torch.autograd.grad(*reversed(_call(x, y)))[0] for y in ys]
  got = [None] * 4
  torch.cuda.synchronize()

  def work(k):
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
      for _ in range(3):
        a, loss = _call(x, ys[k])
        got[k] = torch.autograd.grad(loss, a)[0]
    s.synchronize()
  ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
  for t in ts:
    t.start()
  for t in ts:
    t.join()
  for g, w in zip(got, want):
    assert torch.equal(g, w)
