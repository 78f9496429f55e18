"""Waits between the workgroups of a launch (csrc/waits.h).

A wait that nothing answers must end: the run gives up, spoils its results with
NaN and is reported once, by the next call or by pjz_fdtd_run_status, and the
calls after that are sound again.  The condition is forced from the host
(pjz_fdtd_test_faults: waits end at the first poll in vain); every kernel runs
to its end.  Resident runs of several streams and threads at once must equal
the same runs one after the other.
"""

import threading

import numpy as np
import pytest
import torch

import test_fdtdz_gpu as T
from pjz_amd import _lib
from pjz_amd import _mode as M
from pjz_amd import fdtdz_torch as F

pytestmark = pytest.mark.gpu


class stalled:
  """Calls of this thread inside the block give up waiting at once."""

  def __enter__(self):
    _lib.load().pjz_fdtd_test_faults(_lib.TEST_STALL)

  def __exit__(self, *_):
    _lib.load().pjz_fdtd_test_faults(0)
    torch.cuda.synchronize()


def problem(X, Y, Z, steps=40, axis=0):
  kw = T.random_problem(axis, X=X, Y=Y, Z=Z, tt=steps, seed=X, widths=(6, 5))
  kw["output_steps"] = (steps - 4, steps, 1)
  return kw


def reported():
  """Whether a run has given up since the last report."""
  return _lib.load().pjz_fdtd_run_status() == _lib.ESTALL


# Own polls, polls shared by a workgroup's waves, slabs.
@pytest.mark.parametrize("X,Y,Z", [(64, 64, 64), (128, 128, 64), (150, 140, 96), (260, 196, 96)])
def test_run_that_waits_in_vain_gives_up_and_is_reported_once(X, Y, Z):
  print(f"case {X}x{Y}x{Z}", flush=True)
  kw = problem(X, Y, Z)
  want = F.fdtdz(**kw)
  torch.cuda.synchronize()
  assert not reported()
  with stalled():
    got = F.fdtdz(**kw)
  assert bool(torch.isnan(got).any())
  with pytest.raises(RuntimeError, match="gave up waiting"):
    F.fdtdz(**kw)
  assert not reported()
  assert torch.equal(F.fdtdz(**kw), want)


@pytest.mark.parametrize("X,Y,Z", [(100, 90, 64), (300, 300, 64)])
def test_gradient_that_waits_in_vain(X, Y, Z):
  """The forward is sound, the backward's runs give up."""
  kw = problem(X, Y, Z, steps=50)
  eps = torch.tensor(kw["epsilon"], device="cuda", requires_grad=True)
  kw.update(epsilon=eps, launch_params=dict(ckpt_every=20))

  def grad(fault):
    eps.grad = None
    out = F.fdtdz(**kw)
    ctx = out.grad_fn
    torch.cuda.synchronize()
    if not fault:
      return torch.autograd.grad(out.sum(), eps)[0]
    with stalled():  # (of this thread: autograd's own would not see it)
      g = F._backward(ctx.prob, ctx.dev, ctx.device, ctx.ws, torch.ones_like(out))
    return g

  want = grad(False)
  assert bool(torch.isnan(grad(True)).any())
  assert reported() and not reported()
  # (Cells at the window's border collect their share by atomic additions.)
  torch.testing.assert_close(grad(False), want, rtol=1e-4, atol=1e-5 * float(want.abs().max()))


def test_batch_that_waits_in_vain():
  calls = [problem(128, 120, 64), problem(110, 90, 96), problem(260, 196, 96)]
  want = F.fdtdz_batch(calls)
  with stalled():
    got = F.fdtdz_batch(calls)
  assert all(bool(torch.isnan(o).any()) for o in got)
  with pytest.raises(RuntimeError, match="gave up waiting"):
    F.fdtdz_batch(calls)
  for a, b in zip(F.fdtdz_batch(calls), want):
    assert torch.equal(a, b)


def test_step_by_step_option_does_not_wait():
  for shape in [(128, 128, 64), (260, 196, 96)]:
    kw = dict(problem(*shape), launch_params=dict(resident=False))
    with stalled():
      got = F.fdtdz(**kw)
    assert not reported()
    assert torch.equal(got, F.fdtdz(**dict(kw, launch_params=dict(kernel="stream2"))))


# Frequencies that stop one by one, and together; of several workgroups each.
@pytest.mark.parametrize("X,Y,ww,modes", [(64, 48, 1, 2), (64, 48, 3, 1), (128, 96, 2, 2)])
def test_mode_solve_that_waits_in_vain(X, Y, ww, modes):
  eps = torch.ones(3, X, Y, device="cuda")
  eps[:, X // 3:X // 2, Y // 3:Y // 2] = 12.25
  omega = torch.linspace(0.25, 0.3, ww, device="cuda")
  gen = torch.Generator().manual_seed(X)
  x = torch.randn((ww, 2, X, Y, modes), generator=gen).cuda()
  args = (eps, omega, torch.zeros_like(omega), x, 40, 0.0)
  want = M._subspace_iteration_hip(*args)
  with stalled():
    with pytest.raises(RuntimeError, match="gave up waiting"):
      M._subspace_iteration_hip(*args)
  assert not reported()
  for a, b in zip(M._subspace_iteration_hip(*args)[:3], want):
    assert torch.equal(a, b) and bool(torch.isfinite(a).all())


def test_resident_runs_of_several_streams_and_threads():
  """Each of three threads keeps two streams busy with runs that take the whole
  GPU each; everything as when run one after the other."""
  shapes = [(128, 128, 64), (64, 64, 64), (150, 140, 96)]
  kws = [problem(*s, steps=60, axis=a) for a, s in enumerate(shapes)]
  kws = [{k: torch.as_tensor(v, device="cuda") if isinstance(v, np.ndarray) else v
          for k, v in kw.items()} for kw in kws]
  want = [F.fdtdz(**kw) for kw in kws]
  torch.cuda.synchronize()
  got, errors = [[] for _ in kws], []

  def work(i):
    try:
      streams = [torch.cuda.Stream(), torch.cuda.Stream()]
      for rep in range(4):
        with torch.cuda.stream(streams[rep % 2]):
          got[i].append(F.fdtdz(**kws[i]))
      for s in streams:
        s.synchronize()
    except Exception as e:  # (a thread's exception would be lost)
      errors.append(e)

  threads = [threading.Thread(target=work, args=(i,)) for i in range(len(kws))]
  for t in threads:
    t.start()
  for t in threads:
    t.join()
  torch.cuda.synchronize()
  assert not errors, errors
  for i, w in enumerate(want):
    assert len(got[i]) == 4
    for o in got[i]:
      assert torch.equal(o, w)
  assert not reported()
