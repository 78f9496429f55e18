"""The resident stepper (a whole run in one launch, fields in registers; the
default on domains that fit the registers) against the FP64 oracle (relative
L2 <= 1e-4) and the two-step kernel (<= 1e-6: the same per-cell arithmetic in
the same order of rounding).

Covered: every source axis, one and two cells a lane, odd heights, PML widths
odd, even, one-sided and zero, domains smaller than a tile and with ragged
last tiles, step counts around the shortest resident run, snapshots after
every step, tilings from 2 to 32 cells a lane (cb in registers and from
memory), and the gradient through its checkpoints and recomputes.
"""

import numpy as np
import pytest
import torch

import test_fdtdz_gpu as T
import test_grad_gpu as G
from oracle import c_oracle as C
from pjz_amd import fdtdz_torch as F

pytestmark = pytest.mark.gpu


def run(kw, kernel=None):
  out = F.fdtdz(**dict(kw, launch_params=dict(kernel=kernel) if kernel else None))
  torch.cuda.synchronize()
  return out.cpu().numpy()


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("X,Y,Z,widths", [(22, 19, 24, (5, 4)), (9, 70, 64, (10, 10)),
                                          (61, 17, 33, (0, 7)), (22, 19, 96, (16, 16)),
                                          (19, 33, 99, (6, 5)), (40, 20, 128, (0, 0))])
def test_matches_oracle(X, Y, Z, widths, axis):
  print(f"case {X}x{Y}x{Z} widths={widths} axis={axis}", flush=True)
  kw = T.random_problem(axis, X=X, Y=Y, Z=Z, tt=61, seed=Z + axis, widths=widths)
  kw["output_steps"] = (40, 61, 1)
  got = run(kw)
  assert T.rel_l2(got, C.fdtdz(**kw)) <= T.TOL
  kernel = "stream2" if Z <= 64 or Z % 2 == 0 else "stream"
  assert T.rel_l2(got, run(kw, kernel)) <= 1e-6


@pytest.mark.parametrize("steps", [15, 16, 17])
def test_shortest_runs(steps):
  kw = T.random_problem(0, X=22, Y=19, Z=40, tt=steps, seed=steps, widths=(5, 4))
  kw["output_steps"] = (steps - 2, steps, 1)
  assert T.rel_l2(run(kw), C.fdtdz(**kw)) <= T.TOL


# A domain for each of the tilings: columns a wave x cells a lane.
@pytest.mark.parametrize("X,Y,Z", [(64, 64, 64), (83, 90, 20), (110, 107, 64), (128, 128, 50),
                                   (157, 149, 64), (177, 180, 40), (200, 201, 33),
                                   (222, 230, 45), (301, 187, 45), (250, 255, 24),
                                   (64, 64, 128), (90, 91, 96), (111, 107, 65), (127, 128, 100),
                                   (141, 142, 96), (153, 160, 96), (177, 170, 96),
                                   (180, 182, 66)])
def test_every_tiling_matches_two_step_kernel(X, Y, Z):
  print(f"case {X}x{Y}x{Z}", flush=True)
  kw = T.random_problem(0, X=X, Y=Y, Z=Z, tt=40, seed=X, widths=(6, 5))
  kw["output_steps"] = (30, 40, 3)
  kernel = "stream2" if Z <= 64 or Z % 2 == 0 else "stream"
  assert T.rel_l2(run(kw), run(kw, kernel)) <= 1e-6


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("Z,widths", [(24, (5, 4)), (96, (8, 8)), (99, (5, 6))])
@pytest.mark.parametrize("launch", [{}, dict(ckpt_every=7), dict(ckpt_every=90),
                                    dict(ckpt_every=20, ckpt_inner=7),
                                    dict(ckpt_every=30, ckpt_inner=4)])
def test_gradient_matches_oracle(launch, Z, widths, axis):
  print(f"case {launch} Z={Z} axis={axis}", flush=True)
  eps, kw, g = G.problem(axis, seed=Z + axis, Z=Z, widths=widths)
  ref = G.adjoint.grad_epsilon(eps, g_out=g, **kw)
  got, out = G.gpu_grad(eps, kw, g, **launch)
  assert G.rel_l2(out, C.fdtdz(eps, **kw)) <= T.TOL
  assert G.rel_l2(got, ref) <= G.TOL


def test_gradient_of_a_large_tiling():
  """20 cells a lane (cb from memory) against the two-step kernels."""
  eps, kw, g = G.problem(0, seed=5, X=190, Y=200, Z=50, tt=40)
  g = g * (np.abs(g) > 2)
  got, _ = G.gpu_grad(eps, kw, g, ckpt_every=9)
  ref, _ = G.gpu_grad(eps, kw, g, ckpt_every=9, kernel="stream2")
  assert G.rel_l2(got, ref) <= 1e-5


# Reverse tilings: cb, G and D in registers (2-8 cells a lane), cb from memory
# (12), cb and G from memory (16).
@pytest.mark.parametrize("axis,X,Y,Z", [(0, 64, 62, 33), (1, 83, 90, 20), (2, 110, 107, 24),
                                        (0, 128, 120, 30), (1, 157, 149, 25), (2, 177, 180, 24),
                                        (0, 60, 61, 66), (1, 90, 88, 70), (2, 111, 107, 68),
                                        (0, 128, 126, 66)])
def test_every_reverse_tiling_matches_two_step_kernels(axis, X, Y, Z):
  print(f"case {X}x{Y}x{Z} axis {axis}", flush=True)
  eps, kw, g = G.problem(axis, seed=X, X=X, Y=Y, Z=Z, tt=40)
  got, _ = G.gpu_grad(eps, kw, g, ckpt_every=11)
  ref, _ = G.gpu_grad(eps, kw, g, ckpt_every=11, kernel="stream2")
  assert G.rel_l2(got, ref) <= 1e-5


def test_batch_of_resident_and_streamed_simulations():
  """Each simulation of a batch that mixes both: fields and gradients equal
  its own call's on the two-step kernels."""
  cases = [G.problem(axis, seed=axis, X=X, Y=Y, Z=Z, tt=tt)
           for axis, X, Y, Z, tt in [(0, 130, 120, 64, 40), (1, 30, 40, 64, 41),
                                     (2, 230, 210, 128, 40), (0, 100, 120, 96, 46)]]
  eps = [torch.tensor(e, device="cuda", requires_grad=True) for e, _, _ in cases]
  calls = [dict(kw, epsilon=e, launch_params=dict(ckpt_every=12))
           for e, (_, kw, _) in zip(eps, cases)]
  outs = F.fdtdz_batch(calls)
  sum((o * torch.as_tensor(g, device="cuda")).sum() for o, (_, _, g) in zip(outs, cases)).backward()
  torch.cuda.synchronize()
  plain = F.fdtdz_batch([dict(c, epsilon=c["epsilon"].detach()) for c in calls])
  for e, o, q, (e0, kw, g) in zip(eps, outs, plain, cases):
    ref, out = G.gpu_grad(e0, kw, g, ckpt_every=12, kernel="stream2")
    print(tuple(e.shape), flush=True)
    assert G.rel_l2(o.detach().cpu().numpy(), out) <= 1e-6
    assert G.rel_l2(q.cpu().numpy(), out) <= 1e-6
    assert G.rel_l2(e.grad.cpu().numpy(), ref) <= 1e-5


# Larger domains in slabs of x (two to five), each with ghost columns that a
# block of steps uses up: snapshots inside a block and after it, runs that end
# inside one, every source axis, ragged last slabs.
@pytest.mark.parametrize("axis,X,Y,Z,steps", [(0, 260, 196, 96, 50), (1, 200, 190, 96, 37),
                                              (2, 223, 201, 96, 45), (0, 300, 301, 64, 53),
                                              (2, 401, 300, 45, 41), (0, 129, 341, 128, 40),
                                              (1, 256, 341, 50, 64), (0, 500, 81, 99, 40)])
def test_slabs_match_streaming_kernels(axis, X, Y, Z, steps):
  print(f"case {X}x{Y}x{Z} axis {axis}", flush=True)
  kw = T.random_problem(axis, X=X, Y=Y, Z=Z, tt=steps, seed=X, widths=(6, 5))
  kw["output_steps"] = (steps - 23, steps, 2)
  if axis == 0:
    kw["source_position"] = 2 * (X // 4)  # in the slabs' ghost columns
  kernel = "stream2" if Z <= 64 or Z % 2 == 0 else "stream"
  assert T.rel_l2(run(kw), run(kw, kernel)) <= 1e-6


@pytest.mark.parametrize("launch", [dict(ckpt_every=20), dict(ckpt_every=44, ckpt_inner=18)])
def test_slab_gradient_matches_streaming_kernels(launch):
  eps, kw, g = G.problem(0, seed=9, X=260, Y=196, Z=96, tt=60)
  got, _ = G.gpu_grad(eps, kw, g, **launch)
  ref, _ = G.gpu_grad(eps, kw, g, kernel="stream2", **launch)
  assert G.rel_l2(got, ref) <= 1e-5


def test_batch_with_slabs():
  """As test_batch_of_resident_and_streamed_simulations, with domains in slabs."""
  cases = [G.problem(axis, seed=axis, X=X, Y=Y, Z=Z, tt=tt)
           for axis, X, Y, Z, tt in [(0, 260, 196, 96, 40), (1, 30, 40, 64, 41),
                                     (2, 300, 300, 64, 40)]]
  eps = [torch.tensor(e, device="cuda", requires_grad=True) for e, _, _ in cases]
  calls = [dict(kw, epsilon=e, launch_params=dict(ckpt_every=18))
           for e, (_, kw, _) in zip(eps, cases)]
  outs = F.fdtdz_batch(calls)
  sum((o * torch.as_tensor(g, device="cuda")).sum() for o, (_, _, g) in zip(outs, cases)).backward()
  plain = F.fdtdz_batch([dict(c, epsilon=c["epsilon"].detach()) for c in calls])
  for e, o, q, (e0, kw, g) in zip(eps, outs, plain, cases):
    ref, out = G.gpu_grad(e0, kw, g, ckpt_every=18, kernel="stream2")
    assert G.rel_l2(o.detach().cpu().numpy(), out) <= 1e-6
    assert G.rel_l2(q.cpu().numpy(), out) <= 1e-6
    assert G.rel_l2(e.grad.cpu().numpy(), ref) <= 1e-5
