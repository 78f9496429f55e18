"""Which way a call takes (pjz_fdtd_route_of, pjz_fdtd_batch_routes), asserted
for the domain each kernel is tested on: a change of the dispatch that leaves a
kernel untested fails here instead of passing on another one.

Forward and reverse tilings that no other file reaches, captured runs in slabs
of more than one block, and the batched launches of simulations that would run
resident by default.
"""

import ctypes

import numpy as np
import pytest
import torch

import test_batch_gpu as B
import test_fdtdz_gpu as T
import test_grad_gpu as G
from oracle import c_oracle as C
from pjz_amd import _lib
from pjz_amd import _mode as M
from pjz_amd import fdtdz_torch as F

pytestmark = pytest.mark.gpu


def prob_of(kw, eps=None, **launch):
  shapes = {k: np.shape(v) for k, v in dict(kw, epsilon=kw.get("epsilon", eps)).items()}
  return F.make_problem(shapes["epsilon"], kw["dt"], shapes["source_field"],
                        kw["source_position"], shapes["absorption_mask"], shapes["pml_kappa"],
                        kw["pml_widths"], kw["output_steps"], shapes["source_waveform"][0], False,
                        launch, kw["offset"])


def tiling(r):
  return (r.cells, r.rx, r.ry)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("want,X,Y,Z", [((1, 2, 1), 64, 64, 64), ((1, 2, 2), 88, 88, 64),
                                        ((2, 1, 1), 40, 40, 128), ((2, 2, 1), 62, 58, 120),
                                        ((2, 5, 2), 136, 122, 66)])
def test_forward_tilings(want, X, Y, Z, axis):
  print(f"case {X}x{Y}x{Z} axis {axis}", flush=True)
  kw = T.random_problem(axis, X=X, Y=Y, Z=Z, tt=40, seed=X + axis, widths=(6, 5))
  kw["output_steps"] = (30, 40, 3)
  r = _lib.route(prob_of(kw))
  assert r.kind == _lib.ROUTE_RESIDENT and tiling(r) == want
  step = prob_of(kw, resident=False)
  assert _lib.route(step).kind == _lib.ROUTE_LAUNCHES
  got = F.fdtdz(**kw)
  ref = F.fdtdz(**dict(kw, launch_params=dict(kernel="stream2")))
  assert torch.equal(got, ref)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("want,X,Y,Z", [((1, 2, 1), 64, 64, 64), ((1, 2, 2), 88, 88, 64),
                                        ((2, 1, 1), 40, 40, 128), ((2, 2, 1), 62, 58, 120)])
def test_reverse_tilings(want, X, Y, Z, axis):
  print(f"case {X}x{Y}x{Z} axis {axis}", flush=True)
  eps, kw, g = G.problem(axis, seed=X, X=X, Y=Y, Z=Z, tt=40)
  r = _lib.route(prob_of(kw, eps, ckpt_every=11), backward=True)
  assert r.kind == _lib.ROUTE_RESIDENT and r.reverse == 1 and tiling(r) == want
  got, _ = G.gpu_grad(eps, kw, g, ckpt_every=11)
  ref, _ = G.gpu_grad(eps, kw, g, ckpt_every=11, kernel="stream2")
  assert G.rel_l2(got, ref) <= 1e-5


# Recomputes that capture, in slabs: two cells a lane and one, segments of
# several blocks, and of one and a part.
@pytest.mark.parametrize("want,X,Y,Z,launch", [
    ((1, 5, 5), 300, 300, 64, dict(ckpt_every=50)),
    ((1, 5, 5), 300, 300, 64, dict(ckpt_every=44, ckpt_inner=23)),
    ((2, 4, 3), 200, 180, 66, dict(ckpt_every=30))])
def test_slab_gradients_that_capture(want, X, Y, Z, launch):
  print(f"case {X}x{Y}x{Z} {launch}", flush=True)
  eps, kw, g = G.problem(0, seed=9, X=X, Y=Y, Z=Z, tt=60)
  r = _lib.route(prob_of(kw, eps, **launch), backward=True)
  assert r.kind == _lib.ROUTE_SLABS and tiling(r) == want
  assert launch.get("ckpt_inner", launch["ckpt_every"]) > r.steps
  got, _ = G.gpu_grad(eps, kw, g, **launch)
  ref, _ = G.gpu_grad(eps, kw, g, kernel="stream2", **launch)
  assert G.rel_l2(got, ref) <= 1e-5


def test_three_steps_per_launch_in_batches():
  """Simulations that run resident by default, in the batched launches: the
  zz <= 64 class three steps a launch, uneven step counts (remainders 0, 1, 2),
  snapshots every step at the end."""
  cases = [(11, 150, 140, 64, 60, 0), (12, 130, 150, 40, 50, 1), (13, 141, 122, 64, 49, 2),
           (14, 90, 70, 128, 44, 0)]
  calls = []
  for c in cases:
    kw = B.sim(*c)
    kw["output_steps"] = (c[4] - 7, c[4], 1)
    calls.append(dict(kw, launch_params=dict(resident=False)))
  probs, _, _ = F._batch_problems(calls)
  assert all(r.kind == _lib.ROUTE_LAUNCHES and r.batched for r in _lib.batch_routes(probs))
  probs, _, _ = F._batch_problems([dict(kw, launch_params=None) for kw in calls])
  assert all(r.kind == _lib.ROUTE_RESIDENT and not r.batched for r in _lib.batch_routes(probs))
  outs = F.fdtdz_batch(calls)
  torch.cuda.synchronize()
  for case, kw, out in zip(cases, calls, outs):
    print(f"case {case}", flush=True)
    got = out.cpu().numpy()
    ref = C.fdtdz(**kw)
    assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref), case
    kernel = "stream3" if case[3] <= 64 else "stream2"
    want = F.fdtdz(**dict(kw, launch_params=dict(kernel=kernel))).cpu().numpy()
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want), case


class refused:
  """Cooperative launches of this thread's calls inside the block are refused:
  all, or all but a call's first."""

  def __init__(self, later=False):
    self.fault = _lib.TEST_REFUSE_LATER if later else _lib.TEST_REFUSE

  def __enter__(self):
    _lib.load().pjz_fdtd_test_faults(self.fault)

  def __exit__(self, *_):
    _lib.load().pjz_fdtd_test_faults(0)


@pytest.mark.parametrize("later", [False, True])
@pytest.mark.parametrize("X,Y,Z", [(88, 88, 64), (136, 122, 66), (260, 196, 96), (300, 300, 64)])
def test_refused_launches_step_instead(X, Y, Z, later):
  """A cooperative launch that the runtime refuses leaves the run, or what is
  left of it (slabs), to the kernels launched step by step: the same snapshots."""
  kw = T.random_problem(1, X=X, Y=Y, Z=Z, tt=60, seed=X, widths=(6, 5))
  kw["output_steps"] = (10, 60, 7)
  assert _lib.route(prob_of(kw)).kind != _lib.ROUTE_LAUNCHES
  want = F.fdtdz(**kw)
  with refused(later):
    got = F.fdtdz(**kw)
  assert torch.equal(got, want)
  with refused(later):
    outs = F.fdtdz_batch([kw, kw])
  for o in outs:
    diff = float(torch.linalg.vector_norm(o - want))
    assert diff <= 1e-6 * float(torch.linalg.vector_norm(want))


@pytest.mark.parametrize("later", [False, True])
@pytest.mark.parametrize("launch", [dict(ckpt_every=20), dict(ckpt_every=40, ckpt_inner=18)])
@pytest.mark.parametrize("X,Y,Z", [(88, 88, 64), (124, 136, 66), (300, 300, 64)])
def test_refused_launches_in_gradients(X, Y, Z, launch, later):
  """The same for the recompute and the reverse (refused from the first, or
  from the second launch on: the first segment's reverse)."""
  eps, kw, g = G.problem(0, seed=9, X=X, Y=Y, Z=Z, tt=60)
  assert _lib.route(prob_of(kw, eps, **launch), backward=True).kind != _lib.ROUTE_LAUNCHES
  want, _ = G.gpu_grad(eps, kw, g, **launch)
  out = F.fdtdz(torch.tensor(eps, device="cuda", requires_grad=True),
                **dict(kw, launch_params=launch))
  ctx = out.grad_fn
  with refused(later):  # (of this thread: autograd's own would not see it)
    got = F._backward(ctx.prob, ctx.dev, ctx.device, ctx.ws, torch.as_tensor(g, device="cuda"))
  assert G.rel_l2(got.cpu().numpy(), want) <= 1e-5


def test_refused_launches_in_mode_solves():
  eps = torch.ones(3, 96, 64, device="cuda")
  eps[:, 30:50, 20:40] = 12.25
  omega = torch.tensor([0.25, 0.3], device="cuda")
  x = torch.randn((2, 2, 96, 64, 1), generator=torch.Generator().manual_seed(1)).cuda()
  args = (eps, omega, torch.zeros_like(omega), x, 40, 0.0)
  want = M._subspace_iteration_hip(*args)
  with refused():
    got = M._subspace_iteration_hip(*args)
  for a, b in zip(got[:2], want[:2]):
    torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5)


def test_masked_streams_take_no_launches_that_need_the_whole_gpu():
  """On a stream whose kernels keep to a part of the compute units, workgroups
  that wait for one another might not all run at once."""
  hip = ctypes.CDLL("libamdhip64.so")
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  words = (cus + 31) // 32
  masked = ctypes.c_void_p()
  half = (ctypes.c_uint32 * words)(*[0x0000FFFF] * words)
  assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(masked), words, half) == 0
  try:
    stream = torch.cuda.ExternalStream(masked.value)
    plain = torch.cuda.Stream()
    for X, Y, Z in [(88, 88, 64), (260, 196, 96)]:
      kw = T.random_problem(1, X=X, Y=Y, Z=Z, tt=40, seed=X, widths=(6, 5))
      p = prob_of(kw)
      assert _lib.route(p, stream=masked.value).kind == _lib.ROUTE_LAUNCHES
      assert _lib.route(p, stream=plain.cuda_stream).kind != _lib.ROUTE_LAUNCHES
      want = F.fdtdz(**kw)
      torch.cuda.synchronize()
      with torch.cuda.stream(stream):
        got = F.fdtdz(**kw)
        stream.synchronize()
      assert torch.equal(got, want)
  finally:
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(masked) == 0


def test_batch_in_a_workspace_without_the_slabs_words():
  """Sized for the launches alone, a batch's workspace is enough: its
  simulations in slabs then step as well (single calls: below)."""
  kws = [T.random_problem(1, X=X, Y=Y, Z=Z, tt=40, seed=X, widths=(6, 5))
         for X, Y, Z in [(260, 196, 96), (40, 44, 96)]]
  kws = [dict(kw, output_steps=(20, 40, 7)) for kw in kws]
  probs, devs, device = F._batch_problems(kws)
  lean, _, _ = F._batch_problems([dict(kw, launch_params=dict(resident=False)) for kw in kws])
  small, full = F._batch_workspace_bytes(lean), F._batch_workspace_bytes(probs)
  assert small < full
  want = F.fdtdz_batch(kws)
  outs = [torch.empty_like(o) for o in want]
  ws = F._Workspace(small, device)
  col = lambda j: F._ptrs([d[j] for d in devs])
  rc = _lib.load().pjz_fdtd_batch_forward(
      probs, len(kws), col(0), col(3), col(4), col(5), col(6), col(1), col(2), F._ptrs(outs), ws.ptr,
      ctypes.c_size_t(small), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
  _lib.check(rc, "pjz_fdtd_batch_forward")
  # (35 steps: the odd last one is the one-step kernel's in a single call, the
  # first of a pair's in a batch.)
  for a, b in zip(outs, want):
    diff = float(torch.linalg.vector_norm(a - b))
    assert diff <= 1e-6 * float(torch.linalg.vector_norm(b))
  # The single call of the first.
  p, dev = probs[0], devs[0]
  small = _lib.workspace_bytes(lean[0])
  assert small < _lib.workspace_bytes(p)
  out, ws = torch.empty_like(want[0]), F._Workspace(small, device)
  rc = _lib.load().pjz_fdtd_forward(
      ctypes.byref(p), *[F._ptr(dev[j]) for j in (0, 3, 4, 5, 6, 1, 2)], F._ptr(out), ws.ptr,
      ctypes.c_size_t(small), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
  _lib.check(rc, "pjz_fdtd_forward")
  diff = float(torch.linalg.vector_norm(out - want[0]))
  assert diff <= 1e-6 * float(torch.linalg.vector_norm(want[0]))


def test_mode_solve_in_a_workspace_without_the_tile_kernels_words():
  """A section with few long rows, whose exchange takes more room than the
  other kernels do."""
  X, Y, modes = 32, 512, 1
  nall = 3 * modes + modes * (modes + 1) // 2
  small = 4 * (4 * X * Y * modes + 64 + 32 * nall * 2)
  full = ctypes.c_size_t()
  lib = _lib.load()
  _lib.check(lib.pjz_fdtd_mode_workspace_bytes(1, X, Y, modes, ctypes.byref(full)), "mode")
  assert small < full.value
  eps = torch.ones(3, X, Y, device="cuda")
  eps[:, 10:20, 200:260] = 12.25
  omega, shift = torch.full((1,), 0.25, device="cuda"), torch.zeros(1, device="cuda")
  start = torch.randn((1, 2, X, Y, modes), generator=torch.Generator().manual_seed(1)).cuda()

  def solve(nbytes):
    x, w, err = start.clone(), torch.empty(1, modes, device="cuda"), torch.empty(1, modes,
                                                                                 device="cuda")
    iters = torch.empty(1, dtype=torch.int32, device="cuda")
    ws = torch.empty(nbytes // 4, device="cuda")
    rc = lib.pjz_fdtd_mode_solve(1, X, Y, modes, *[F._ptr(t) for t in
                                                  (eps, omega, shift, x, w, err, iters)], 40, 0.0,
                                 F._ptr(ws), nbytes,
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return rc, w, x

  assert solve(small - 4)[0] == _lib.ESPACE
  rc, w, x = solve(small)
  _lib.check(rc, "mode")
  rc, w1, x1 = solve(full.value)
  _lib.check(rc, "mode")
  torch.testing.assert_close(w, w1, rtol=1e-4, atol=1e-5)
  torch.testing.assert_close(x, x1, rtol=1e-3, atol=1e-4)


@pytest.mark.parametrize("many", [2, 3])
def test_batched_gradients_share_launches_unless_their_recompute_is_resident(many):
  """Forward alone, backward batched, of three simulations whose tiling cannot
  capture (two cells a lane past 25); alone where there are only two, and where
  it can, with and without a resident reverse."""
  cases = [(180, 150, 128), (150, 140, 96), (128, 120, 64)] + [(170, 150, 96)] * (many - 1)
  probs = [G.problem(0, seed=i, X=X, Y=Y, Z=Z, tt=40) for i, (X, Y, Z) in enumerate(cases)]
  eps = [torch.tensor(e, device="cuda", requires_grad=True) for e, _, _ in probs]
  calls = [dict(kw, epsilon=e, launch_params=dict(ckpt_every=12))
           for e, (_, kw, _) in zip(eps, probs)]
  ps, _, _ = F._batch_problems(calls)
  assert [r.kind for r in _lib.batch_routes(ps)] == [_lib.ROUTE_RESIDENT] * len(cases)
  back = _lib.batch_routes(ps, backward=True)
  assert [r.kind for r in back[1:3]] == [_lib.ROUTE_RESIDENT] * 2
  assert [r.reverse for r in back[:3]] == [0, 0, 1]
  assert [r.batched for r in back] == [many == 3, False, False] + [many == 3] * (many - 1)
  outs = F.fdtdz_batch(calls)
  sum((o * torch.as_tensor(g, device="cuda")).sum() for o, (_, _, g) in zip(outs, probs)).backward()
  torch.cuda.synchronize()
  for e, o, (e0, kw, g) in zip(eps, outs, probs):
    print(tuple(e.shape), flush=True)
    ref, out = G.gpu_grad(e0, kw, g, ckpt_every=12, kernel="stream2")
    assert G.rel_l2(o.detach().cpu().numpy(), out) <= 1e-6
    assert G.rel_l2(e.grad.cpu().numpy(), ref) <= 1e-5


@pytest.mark.parametrize("X,Y,Z", [(64, 64, 64), (260, 196, 96)])
def test_recorded_calls_are_launched_step_by_step(X, Y, Z):
  """A call recorded into a graph makes no cooperative launch and allocates no
  host memory; its replays, with eager runs in between, equal those."""
  kw = T.random_problem(1, X=X, Y=Y, Z=Z, tt=40, seed=X, widths=(6, 5))
  prob = prob_of(kw)
  kw = {k: torch.as_tensor(v, device="cuda") if isinstance(v, np.ndarray) else v
        for k, v in kw.items()}
  want = F.fdtdz(**kw)
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    route = _lib.route(prob, stream=torch.cuda.current_stream().cuda_stream)
    out = F.fdtdz(**kw)
  assert route.kind == _lib.ROUTE_LAUNCHES
  for _ in range(3):
    out.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    assert torch.equal(F.fdtdz(**kw), want)
    torch.cuda.synchronize()
