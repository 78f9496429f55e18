"""The workloads the framework is timed on, with float64 results to check them.

Each case is one call (or one call and its gradient) through the package's
public entry points, at sizes its tests, workloads and benchmark use or that
lie between them.  ``listed()`` names them, ``draw()`` gives more of the same
ranges, ``prepare()`` builds the inputs on the GPU from a seed, ``run()`` makes
one pass and ``exact()`` computes the same outputs in float64 with plain torch
operations only.
"""

import math

import numpy as np
import torch

import pjz_amd
from pjz_amd import boundaries as B


def _device():
  return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------ the cases
def listed():
  return [
      # The smallest simulation in use: a 64^3 layered stack over its 2000
      # steps.  Every step is a launch or less, so latency counts.
      dict(name="forward_64", kind="forward", xx=64, yy=64, zz=64, lo=10, hi=10, axis=0,
           steps=2000, stack="layers", amount=1),
      # The headline simulation, 512x512x128 with a 200x200 design region, over
      # the first part of its run: fields far larger than the caches.
      dict(name="forward_512", kind="forward", xx=512, yy=512, zz=128, lo=16, hi=16, axis=0,
           steps=600, stack="design", amount=1),
      # Nothing a multiple of anything: odd sizes, unequal PML, a z-plane source.
      dict(name="forward_ragged", kind="forward", xx=301, yy=187, zz=45, lo=9, hi=12, axis=2,
           steps=600, stack="design", amount=1),
      # field() with default parameters (50 absorber cells a side, height 96)
      # on a mid-sized structure and two frequencies: host glue, a simulation
      # and the projection.
      dict(name="field_default", kind="field", xx=120, yy=100, zz=40, steps=800, ww=2),
      # The gradient workload's 256x256x128 grid: a simulation with its
      # checkpoints and the adjoint.
      dict(name="gradient_256", kind="gradient", xx=256, yy=256, zz=128, lo=10, hi=10, axis=0,
           steps=300, stack="layers", amount=1),
      # One design variant by itself: a small simulation with its gradient.
      dict(name="gradient_128", kind="gradient", xx=128, yy=128, zz=64, lo=10, hi=10, axis=0,
           steps=600, stack="design", amount=1),
      # An uneven batch, forward only.
      dict(name="batch_uneven", kind="batch", xx=128, yy=384, zz=128, lo=10, hi=10, axis=0,
           steps=300, stack="design", amount=6),
      # An inverse-design iteration's batch: equal simulations with gradients.
      dict(name="batch_design", kind="batch_gradient", xx=128, yy=128, zz=64, lo=10, hi=10, axis=0,
           steps=400, stack="design", amount=8),
      # Scattering parameters of a two-port device and their gradient.
      dict(name="scatter_2port", kind="scatter", xx=160, yy=96, zz=24, steps=500, ww=2),
      # Port modes: the small strip and the large cross-section.
      dict(name="mode_30x20", kind="mode", xx=30, yy=20, ww=1, modes=2, iters=1500),
      dict(name="mode_256x128", kind="mode", xx=256, yy=128, ww=1, modes=2, iters=500),
      # From the design variable to the permittivity and back: the density
      # filter, the layered render and both reverse passes.
      dict(name="design_384", kind="design", xx=384, yy=384, zz=128, m=2, radius=6.0),
  ]


def _log(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  kind = rng.choice(["forward", "forward", "forward", "field", "gradient", "gradient", "batch",
                     "batch_gradient", "scatter", "mode", "mode", "design"])
  if kind == "mode":
    xx, yy = _log(rng, 20, 256), _log(rng, 16, 128)
    return dict(kind=kind, xx=xx, yy=yy, ww=rng.choice([1, 1, 2, 3]), modes=rng.choice([1, 2, 2, 3]),
                iters=_log(rng, 200, 1500) if xx * yy < 4000 else _log(rng, 150, 500))
  if kind == "design":
    return dict(kind=kind, xx=_log(rng, 32, 384), yy=_log(rng, 32, 384), zz=_log(rng, 16, 128),
                m=rng.choice([1, 2, 2, 3]), radius=rng.choice([1.5, 3.0, 4.0, 6.0, 8.5]))
  if kind in ("field", "scatter"):
    return dict(kind=kind, xx=_log(rng, 48, 160), yy=_log(rng, 40, 120), zz=_log(rng, 12, 60),
                steps=_log(rng, 300, 800) if kind == "field" else _log(rng, 300, 500),
                ww=rng.choice([1, 2]))
  # Cells times steps of the largest listed case of the kind bound a draw.
  most = {"forward": 2.0e10, "gradient": 2.5e9, "batch": 2.4e9, "batch_gradient": 2.5e9}[kind]
  xx, yy = _log(rng, 40, 512 if kind == "forward" else 256), _log(rng, 40, 512 if kind == "forward"
                                                                  else 256)
  zz = rng.choice([rng.randint(24, 64), 64, rng.randint(65, 128), 96, 128])
  if kind in ("batch", "batch_gradient"):
    zz += zz % 2
  lo, hi = rng.choice([(10, 10), (16, 16), (10, 10), (8, 11)])
  if lo + hi + 8 > zz:
    lo, hi = 6, 6
  amount = 1 if kind in ("forward", "gradient") else rng.randint(2, 8)
  steps = _log(rng, 200, 2000 if kind == "forward" else 600)
  steps = max(120, min(steps, int(most / (xx * yy * zz * amount))))
  axis = rng.choice([0, 0, 1, 2])
  return dict(kind=kind, xx=xx, yy=yy, zz=zz, lo=lo, hi=hi, axis=axis, steps=steps,
              stack=rng.choice(["layers", "design"]), amount=amount)


# ------------------------------------------------------------------ the inputs
def _gen(seed, salt=0):
  return torch.Generator(device=_device()).manual_seed(1000 * seed + salt)


def _uniform(shape, lo, hi, gen):
  return lo + (hi - lo) * torch.rand(shape, generator=gen, device=gen.device)


def _structure(X, Y, Z, stack, gen):
  """SiO2 below, a Si strip along x in the core, air above; "design" adds a
  centred Bernoulli(0.5) region in the core, "layers" small noise."""
  eps = torch.ones((3, X, Y, Z), device=gen.device)
  z0, z1 = (3 * Z) // 8, max((3 * Z) // 8 + 1, Z // 2)
  eps[..., :z0] = 2.085
  y0, y1 = (13 * Y) // 32, (19 * Y) // 32
  eps[:, :, y0:y1, z0:z1] = 12.25
  if stack == "design":
    dx, dy = X // 5, Y // 5
    pattern = torch.where(torch.rand((2 * dx, 2 * dy), generator=gen, device=gen.device) < 0.5,
                          2.085, 12.25)
    cx, cy = X // 2, Y // 2
    eps[:, cx - dx:cx + dx, cy - dy:cy + dy, z0:z1] = pattern[None, :, :, None]
  else:
    eps += _uniform(eps.shape, -0.01, 0.01, gen)
  return eps


def _bump(n, centre, width, dev):
  return torch.exp(-((torch.arange(n, device=dev) - centre) / width) ** 2 / 2)


def _call(case, X, Y, Z, seed, salt=0):
  """Keyword arguments of one fdtdz() call and the monitor (axis, position,
  profile) its objective uses."""
  gen = _gen(seed, salt)
  dev, axis, steps = gen.device, case["axis"], case["steps"]
  eps = _structure(X, Y, Z, case["stack"], gen)
  n = [X, Y, Z]
  centre = [X / 2, Y / 2, 7 * Z / 16]
  width = [max(3.0, X / 16), max(3.0, Y / 16), max(2.0, Z / 20)]
  line = [_bump(n[a], centre[a] + float(_uniform((), -1, 1, gen)), width[a], dev) for a in range(3)]
  shape = [X, Y, Z]
  shape[axis] = 1
  a, b = [k for k in range(3) if k != axis]
  profile = (line[a][:, None] * line[b][None, :]).reshape(shape)
  source = torch.stack([profile, 0.1 * profile]) * (
      1 + 0.05 * torch.randn([2] + shape, generator=gen, device=dev))
  pos = (7 * Z) // 16 if axis == 2 else 2 * max(6, n[axis] // 16)
  # The monitor: as far as a wave in the core gets, inside the absorber.
  far = pos + 3 if axis == 2 else min(n[axis] - 1 - max(12, n[axis] // 8), pos + steps // 10)
  omegas = np.array([2 * math.pi / 18, 2 * math.pi / 22])
  wave = np.zeros((steps, 2), np.float32)
  wave[:, 0] = np.imag(B.ramped_sin(omegas, 4.0, 2.0, 0.5, steps))
  if axis == 2:
    source = torch.stack([source, 0.5 * source])  # two quadratures
    wave[:, 1] = np.real(B.ramped_sin(omegas, 4.0, 2.0, 0.5, steps))
  pad = min(32, max(6, min(X, Y) // 8))
  f32 = lambda v: torch.as_tensor(np.ascontiguousarray(v, np.float32), device=dev)
  kw = dict(
      epsilon=eps, dt=0.5, source_field=source.contiguous(), source_waveform=f32(wave),
      source_position=pos, absorption_mask=f32(B.absorption_mask(X, Y, pad, 0.1 / pad ** 2)),
      pml_kappa=torch.ones((Z, 2), device=dev),
      pml_sigma=f32(B.pml_sigma((case["lo"], case["hi"]), Z, 0.5, 2.0)),
      pml_alpha=torch.full((Z, 2), 0.05, device=dev), pml_widths=(case["lo"], case["hi"]),
      output_steps=(steps - 16, steps, 5), use_reduced_precision=False, launch_params=None,
      offset=(0, 0, 0))
  return kw, (axis, far, profile)


def _sizes(case):
  """(X, Y, Z) of each simulation of a case: the uneven batch's sides lie
  between its xx and yy, and every other one has half the height."""
  X, Y, Z = case["xx"], case["yy"], case["zz"]
  if case["kind"] != "batch":
    return [(X, Y, Z)] * case["amount"]
  n, out = case["amount"], []
  for i in range(n):
    f, g = ((3 * i) % n) / n, ((2 * i + 1) % n) / n
    z = Z if i % 2 == 0 or Z < 96 else (Z // 4) * 2
    out.append((int(X + f * (Y - X)), int(X + g * (Y - X)), z))
  return out


def _objective(out, monitor, weight):
  """sum over snapshots of (overlap with the monitor's profile)^2: the real
  field form of a mode-overlap objective."""
  axis, pos, profile = monitor
  comps = [c for c in range(3) if c != axis]
  plane = out[:, comps].narrow(2 + axis, pos, 1)
  ov = torch.sum(plane * profile.to(plane.dtype), dim=(1, 2, 3, 4))
  return weight * torch.sum(ov ** 2)


def _field_inputs(case, seed):
  gen = _gen(seed)
  dev = gen.device
  X, Y, Z = case["xx"], case["yy"], case["zz"]
  eps = _structure(X, Y, Z, "design", gen)
  omega = np.array([2 * math.pi / 18, 2 * math.pi / 22])[:case["ww"]]
  line_y, line_z = _bump(Y, Y / 2, max(3.0, Y / 16), dev), _bump(Z, 7 * Z / 16, max(2.0, Z / 10), dev)
  profile = (line_y[:, None] * line_z[None, :])[None]
  noise = lambda: 1 + 0.05 * torch.randn((2, 1, Y, Z), generator=gen, device=dev)
  mode = lambda: torch.stack([profile, 0.1 * profile]) * noise()
  params = pjz_amd.SimParams(omega_range=(float(omega.min()), float(omega.max())),
                             tt=case["steps"])
  return eps, omega, mode, params, max(4, X // 8)


def _section(case, seed):
  """(3, xx, yy) cross-section: a Si strip in SiO2 with small index noise."""
  gen = _gen(seed)
  X, Y = case["xx"], case["yy"]
  eps = torch.full((3, X, Y), 2.085, device=gen.device)
  eps[:, (3 * X) // 10:(7 * X) // 10, (2 * Y) // 5:(3 * Y) // 5] = 12.25
  return eps + _uniform(eps.shape, -0.01, 0.01, gen)


def prepare(case, seed):
  kind, state = case["kind"], dict(case=case)
  if kind in ("forward", "gradient", "batch", "batch_gradient"):
    calls = [_call(case, *size, seed, salt) for salt, size in enumerate(_sizes(case))]
    state.update(calls=[c for c, _ in calls], monitors=[m for _, m in calls])
    state["weight"] = 1.0
    if "gradient" in kind:
      for kw in state["calls"]:
        kw["epsilon"].requires_grad_(True)
  elif kind == "field":
    eps, omega, mode, params, pos = _field_inputs(case, seed)
    state.update(eps=eps, omega=omega, mode=mode(), params=params, pos=pos)
  elif kind == "scatter":
    eps, omega, mode, params, pos = _field_inputs(case, seed)
    modes = [torch.stack([mode() for _ in omega]) for _ in range(2)]
    betas = [torch.as_tensor(2.2 * omega, device=eps.device) for _ in range(2)]
    eps.requires_grad_(True)
    state.update(eps=eps, omega=omega, modes=modes, betas=betas,
                 pos=(pos, case["xx"] - 1 - pos), fwd=(True, False), params=params)
  elif kind == "mode":
    eps = _section(case, seed)
    omega = torch.as_tensor(2 * math.pi / np.linspace(19, 21, 2 * case["ww"] + 1)[1::2],
                            device=eps.device)
    state.update(eps=eps[:, None], omega=omega)  # propagation along x
  elif kind == "design":
    gen = _gen(seed)
    X, Y, Z, m = case["xx"], case["yy"], case["zz"], case["m"]
    # A design part-way through its optimisation: features of tens of pixels,
    # not yet flat inside, and small noise.
    coarse = _uniform((1, 1, 2 + 2 * m * X // 32, 2 + 2 * m * Y // 32), 0, 1, gen)
    u = torch.nn.functional.interpolate(coarse, (2 * m * X, 2 * m * Y), mode="bicubic")[0, 0]
    u = 0.5 + 0.8 * (u - 0.5) + _uniform(u.shape, -0.1, 0.1, gen)
    u = u.contiguous().requires_grad_(True)
    pos = torch.tensor([0.37 * Z, 0.55 * Z], device=gen.device, requires_grad=True)
    state.update(u=u, pos=pos, g_eps=torch.randn((3, X, Y, Z), generator=gen, device=gen.device),
                 g_loss=torch.rand(u.shape, generator=gen, device=gen.device))
  else:
    raise ValueError(kind)
  return state


# ------------------------------------------------------------------ one pass
def _layers(dens):
  """SiO2 below, the design between SiO2 and Si, air above."""
  return torch.stack([torch.full_like(dens, 2.085), 2.085 + (12.25 - 2.085) * dens,
                      torch.ones_like(dens)])


def run(state):
  case = state["case"]
  kind = case["kind"]
  if kind == "forward":
    return pjz_amd.fdtdz(**state["calls"][0])
  if kind == "batch":
    return pjz_amd.fdtdz_batch(state["calls"])
  if kind == "gradient":
    kw = state["calls"][0]
    out = pjz_amd.fdtdz(**kw)
    loss = _objective(out, state["monitors"][0], state["weight"])
    grad, = torch.autograd.grad(loss, kw["epsilon"])
    return out.detach(), loss.detach(), grad
  if kind == "batch_gradient":
    for kw in state["calls"]:
      kw["epsilon"].grad = None
    loss = pjz_amd.fdtdz_batch_value_and_grad(
        state["calls"], lambda i, out: _objective(out, state["monitors"][i], state["weight"]))
    return [loss] + [kw["epsilon"].grad for kw in state["calls"]]
  if kind == "field":
    return pjz_amd.field(state["eps"], state["mode"], state["omega"], state["pos"],
                         state["params"])
  if kind == "scatter":
    s = pjz_amd.scatter(state["eps"], state["omega"], state["modes"], state["betas"],
                        state["pos"], state["fwd"], state["params"])
    s = torch.stack([torch.stack(row) for row in s])
    # Transmission up, reflection down.
    loss = torch.sum(torch.abs(s[0, 0]) ** 2) - torch.sum(torch.abs(s[0, 1]) ** 2)
    grad, = torch.autograd.grad(loss, state["eps"])
    # Overlaps of float32 fields: complex64 holds what they are worth.
    return s.detach().to(torch.complex64), grad
  if kind == "mode":
    # A fixed number of iterations, as an optimisation loop's budget; the
    # residuals are not returned: those of a converged mode are rounding noise.
    beta, exc, _, iters = pjz_amd.mode(state["eps"], state["omega"], case["modes"],
                                       max_iters=case["iters"], tol=0.0)
    return beta, exc, iters
  if kind == "design":
    dens, loss = pjz_amd.density(state["u"], case["radius"], 0.5)
    eps = pjz_amd.epsilon(_layers(dens), state["pos"], case["m"], case["zz"])
    gu, gp = torch.autograd.grad([eps, loss], [state["u"], state["pos"]],
                                 [state["g_eps"], state["g_loss"]])
    return dens.detach(), loss.detach(), eps.detach(), gu, gp
  raise ValueError(kind)


# ------------------------------------------------------------------ what a pass needs
# Floating operations a cell and step: 6 components, a curl of two
# differences (3), the update (2 for H, 3 for E); the adjoint step the same
# and the accumulation (2 a component).
_STEP_FLOPS, _ADJOINT_FLOPS = 33, 39


def work(case):
  kind = case["kind"]
  if kind in ("forward", "gradient", "batch", "batch_gradient"):
    nbytes = flops = 0
    for X, Y, Z in _sizes(case):
      cells, nn = X * Y * Z, 4
      grad = "gradient" in kind
      nbytes += 12 * cells + 12 * nn * cells + 12 * X * Y + (12 * cells if grad else 0)
      # The adjoint needs the forward fields again: its own steps only.
      flops += cells * case["steps"] * (_STEP_FLOPS + (_ADJOINT_FLOPS if grad else 0))
    return {"bytes": nbytes, "flops": flops}
  if kind in ("field", "scatter"):
    X, Y, Z, ww = case["xx"], case["yy"], case["zz"], case["ww"]
    ports = 2 if kind == "scatter" else 1
    cells = (X + 100) * (Y + 100) * 96
    nbytes = 12 * X * Y * Z + (24 * ww * X * Y * Z if kind == "field" else 12 * X * Y * Z)
    return {"bytes": nbytes, "flops": ports * cells * case["steps"] * _STEP_FLOPS}
  if kind == "mode":
    X, Y, mm = case["xx"], case["yy"], case["modes"]
    # The operator (22 a cell and mode), Rayleigh sums (12), orthogonalisation.
    per = mm * (22 + 12) + 2 * mm * mm * 4
    return {"bytes": 4 * case["ww"] * (3 * X * Y + 2 * X * Y * mm),
            "flops": case["ww"] * X * Y * per * case["iters"]}
  X, Y, Z, m = case["xx"], case["yy"], case["zz"], case["m"]
  sub, cells = 4 * m * m * X * Y, X * Y * Z
  # The variable in, density and loss out, cotangent of the loss in and
  # gradient out; the permittivity out and its cotangent in; the blur's and
  # its transpose's taps.
  return {"bytes": 4 * (5 * sub + 6 * cells),
          "flops": sub * 4 * (2 * math.ceil(case["radius"] - 0.5) + 1) ** 2 + cells * 3 * 60}


# ------------------------------------------------------------------ float64
def _dif(f, axis, forward):
  """f[i+1] - f[i] (or f[i] - f[i-1]) with zeros outside."""
  n = f.shape[axis]
  d = f.narrow(axis, 1, n - 1) - f.narrow(axis, 0, n - 1)
  edge = -f.narrow(axis, n - 1, 1) if forward else f.narrow(axis, 0, 1)
  return torch.cat([d, edge] if forward else [edge, d], dim=axis)


class _Exact:
  """The Yee update of one fdtdz() call in float64 torch operations."""

  def __init__(self, kw):
    f64 = lambda a: torch.as_tensor(a).detach().to(torch.float64)
    self.dt = float(kw["dt"])
    mask, eps = f64(kw["absorption_mask"]), f64(kw["epsilon"])
    dev = eps.device
    self.size = (mask.shape[1], mask.shape[2], kw["pml_sigma"].shape[0])
    self.window = tuple(kw["offset"]), tuple(eps.shape[1:])
    self.mask = mask[..., None]
    self.index = [torch.clamp(torch.arange(n, device=dev) - o, 0, e - 1)
                  for n, o, e in zip(self.size, *self.window)]
    self.lo, self.hi = kw["pml_widths"]
    Z = self.size[2]
    kappa, sigma, alpha = (f64(kw[k]).to(dev) for k in ("pml_kappa", "pml_sigma", "pml_alpha"))
    self.ik = 1 / kappa  # 0 for kappa = inf
    damp = sigma * self.ik + alpha
    b = torch.exp(-damp * self.dt)
    c = torch.where((sigma == 0) | (self.ik == 0), torch.zeros_like(b),
                    sigma * self.ik ** 2 * (b - 1) / torch.where(damp == 0, 1.0, damp))
    keep = torch.cat([torch.arange(self.lo), torch.arange(Z - self.hi, Z)]).to(dev)
    self.b, self.c = b[keep], c[keep]
    self.wave = f64(kw["source_waveform"]).cpu().tolist()
    src, p = f64(kw["source_field"]), int(kw["source_position"])
    self.axis = 2 if src.ndim == 5 or src.shape[3] == 1 else 0 if src.shape[1] == 1 else 1
    self.src, self.pos = src if src.ndim == 5 else src[None], p
    r = range(*kw["output_steps"])
    self.want, self.steps = set(r), r[-1] + 1
    self.eps = eps

  def coefficients(self, eps):
    full = eps[:, self.index[0]][:, :, self.index[1]][..., self.index[2]]
    q = self.mask * self.dt / (2 * full)
    return (1 - q) / (1 + q), self.dt / full / (1 + q)

  def start(self):
    z = lambda *s: torch.zeros(s, dtype=torch.float64, device=self.eps.device)
    return [z(*self.size) for _ in range(6)] + [
        z(self.size[0], self.size[1], self.lo + self.hi) for _ in range(4)]

  def _dz(self, f, psi, col):
    """d/dz with its PML: (derivative, new psi)."""
    d = _dif(f, 2, col == 1)
    Z, lo, hi = self.size[2], self.lo, self.hi
    psi = self.b[:, col] * psi + self.c[:, col] * torch.cat([d[..., :lo], d[..., Z - hi:]], 2)
    t = self.ik[:, col] * d
    return torch.cat([t[..., :lo] + psi[..., :lo], t[..., lo:Z - hi],
                      t[..., Z - hi:] + psi[..., lo:]], 2), psi

  def step(self, state, ca, cb, n):
    ex, ey, ez, hx, hy, hz, p0, p1, p2, p3 = state
    dt = self.dt
    zy, p0 = self._dz(ey, p0, 1)
    zx, p1 = self._dz(ex, p1, 1)
    hx = hx - dt * (_dif(ez, 1, True) - zy)
    hy = hy - dt * (zx - _dif(ez, 0, True))
    hz = hz - dt * (_dif(ey, 0, True) - _dif(ex, 1, True))
    zy, p2 = self._dz(hy, p2, 0)
    zx, p3 = self._dz(hx, p3, 0)
    curl = [_dif(hz, 1, False) - zy, zx - _dif(hz, 0, False),
            _dif(hy, 0, False) - _dif(hx, 1, False)]
    comps = [k for k in range(3) if k != self.axis]
    for k, comp in enumerate(comps):
      if self.axis == 2:
        for q in range(self.src.shape[0]):
          curl[comp][:, :, self.pos] += self.src[q, k][..., 0] * self.wave[n][q]
      else:
        for col in (0, 1):
          if self.wave[n][col]:
            curl[comp].narrow(self.axis, self.pos - col, 1).add_(self.src[0, k] *
                                                                 self.wave[n][col])
    e = [ca[k] * f + cb[k] * curl[k] for k, f in enumerate((ex, ey, ez))]
    return e + [hx, hy, hz, p0, p1, p2, p3]

  def snapshot(self, state):
    (x, y, z), (a, b, c) = self.window
    return torch.stack([f[x:x + a, y:y + b, z:z + c] for f in state[:3]])

  @torch.no_grad()
  def forward(self, every=None):
    """Snapshots, and the states before every ``every``-th step."""
    ca, cb = self.coefficients(self.eps)
    state, outs, kept = self.start(), [], []
    for n in range(self.steps):
      if every and n % every == 0:
        kept.append(state)
      state = self.step(state, ca, cb, n)
      if n in self.want:
        outs.append(self.snapshot(state))
    return torch.stack(outs), kept

  def gradient(self, objective):
    """(snapshots, loss, dloss/depsilon), segment by segment with autograd."""
    cells = self.size[0] * self.size[1] * self.size[2]
    every = max(2, min(25, int(4e9 / (70 * 8 * cells) * 8)))
    outs, kept = self.forward(every)
    leaf = outs.clone().requires_grad_(True)
    loss = objective(leaf)
    g_out, = torch.autograd.grad(loss, leaf)
    eps = self.eps.clone().requires_grad_(True)
    ca0, cb0 = self.coefficients(eps)
    ca, cb = ca0.detach().requires_grad_(True), cb0.detach().requires_grad_(True)
    slots = {s: i for i, s in enumerate(sorted(self.want))}
    g_ca, g_cb = torch.zeros_like(ca), torch.zeros_like(cb)
    g_state = [torch.zeros_like(f) for f in kept[0]]
    for k in reversed(range(len(kept))):
      begin = [f.requires_grad_(True) for f in kept.pop()]
      state, heads, cots = begin, [], []
      for n in range(k * every, min((k + 1) * every, self.steps)):
        state = self.step(state, ca, cb, n)
        if n in slots:
          heads.append(self.snapshot(state))
          cots.append(g_out[slots[n]])
      got = torch.autograd.grad(heads + list(state), [ca, cb] + begin, cots + g_state,
                                allow_unused=True)
      g_ca += got[0]
      g_cb += got[1]
      g_state = [torch.zeros_like(f) if g is None else g for g, f in zip(got[2:], begin)]
      del state, begin, heads, got
    grad, = torch.autograd.grad([ca0, cb0], eps, [g_ca, g_cb])
    return outs, loss.detach(), grad


def _exact_glue(state, source, pos):
  """The fdtdz() call that field() makes for one source, built here in float64."""
  eps, p, omega = state["eps"].detach(), state["params"], state["omega"]
  X, Y, Z = eps.shape[1:]
  pad, ZZ = p.absorption_padding, 128 - sum(p.pml_widths)
  dev, ww = eps.device, len(omega)
  bot = (ZZ - Z) // 2
  t = omega[:, None] * p.dt * np.arange(p.tt)
  ramp = (1 + np.tanh(t / p.source_ramp - p.source_delay)) / 2
  wave = np.zeros((p.tt, 2))
  wave[:, 0] = np.mean(ramp * np.sin(t), axis=0)
  period = 4 * math.pi / (omega.max() + omega.min()) / p.dt
  if ww == 1:
    interval = int(round(period / 4))
  else:
    cutoff = math.pi * (ww - 1) / ww / (omega.max() - omega.min()) / p.dt
    interval = int(round(period / 4 + math.floor((cutoff - period / 4) / (period / 2)) *
                         period / 2))
  steps = (p.tt - 2 * interval * ww - 1, p.tt, interval)
  src = source.to(torch.float64) / eps[1:, pos:pos + 1].to(torch.float64)
  src = torch.nn.functional.pad(src, (bot, ZZ - Z - bot, pad, pad))
  at = pos + pad
  if at % 2:
    at, wave = at + 1, wave[:, ::-1].copy()
  ramps = []
  for n in (X + 2 * pad, Y + 2 * pad):
    q = np.arange(n)[None, :] + np.array([[0.0], [0.5]])
    ramps.append(p.absorption_coeff * np.clip(np.abs(q - (n - 1) / 2) - (n - 1) / 2 + pad, 0,
                                              None) ** 2)
  x, y = ramps
  mask = np.stack([np.maximum(x[i][:, None], y[j][None, :]) for i, j in ((0, 1), (1, 0), (1, 1))])
  lo, hi = p.pml_widths
  z = np.arange(ZZ)[:, None] + np.array([[0.0, 0.5]])
  depth = np.clip(np.maximum((lo - z) / lo, (z + 0.5 - ZZ + hi) / hi), 0, None)
  sigma = (p.pml_sigma_m + 1) * p.pml_sigma_lnr * depth ** p.pml_sigma_m
  f64 = lambda v: torch.as_tensor(v, dtype=torch.float64, device=dev)
  kw = dict(epsilon=eps, dt=p.dt, source_field=src, source_waveform=f64(wave), source_position=at,
            absorption_mask=f64(mask), pml_kappa=f64(np.ones((ZZ, 2))), pml_sigma=f64(sigma),
            pml_alpha=f64(np.zeros((ZZ, 2))), pml_widths=p.pml_widths, output_steps=steps,
            offset=(pad, pad, bot))
  theta = omega[:, None] * p.dt * np.arange(*steps)[None, :]
  inverse = f64(np.linalg.pinv(np.concatenate([np.cos(theta), -np.sin(theta)]).T))
  outs, _ = _Exact(kw).forward()
  parts = (inverse @ outs.reshape(outs.shape[0], -1)).reshape((2 * ww,) + outs.shape[1:])
  return torch.complex(parts[:ww], parts[ww:])


def _exact_scatter(state):
  eps, omega = state["eps"].detach(), state["omega"]
  fields = [_exact_glue(state, m.mean(dim=0), p) for m, p in zip(state["modes"], state["pos"])]

  def overlap(mode, beta, pos, fwd, f):
    x = (1.0, 2.0) if fwd else (-2.0, -1.0)
    beta = beta if fwd else -beta
    vals = torch.stack([torch.sum(mode.to(torch.complex128) * f[:, 1:, pos + int(s)][:, :, None],
                                  dim=(1, 2, 3, 4)) for s in x], dim=-1)
    out = []
    for w in range(len(omega)):
      a = torch.tensor([[np.exp(-1j * float(beta[w]) * s) for s in x],
                        [np.exp(1j * float(beta[w]) * s) for s in x]], dtype=torch.complex128)
      out.append(torch.linalg.solve(a.T, vals[w].cpu()).to(eps.device))
    return torch.stack(out)

  ports = list(zip(state["modes"], state["betas"], state["pos"], state["fwd"]))
  amps = [overlap(*p, f)[:, 0] for p, f in zip(ports, fields)]
  s = torch.stack([torch.stack([overlap(*p, f)[:, 1] / a for p in ports])
                   for a, f in zip(amps, fields)])
  # The reciprocity gradient sum Re(conj(g_ij) f_i f_j / a_i), where g_ij is
  # the cotangent dL/dRe + i dL/dIm = 2 s for |s|^2.
  grad = torch.zeros(eps.shape, dtype=torch.float64, device=eps.device)
  for j, sign in ((0, 1.0), (1, -1.0)):
    g = torch.conj(2 * sign * s[0, j]) / amps[0]
    grad += torch.real(torch.sum(g[:, None, None, None, None] * fields[0] * fields[j], dim=0))
  return s, grad


def _exact_mode(case, state):
  f64 = torch.float64
  eps = state["eps"][:, 0].to(f64)[[1, 2, 0]]  # propagation along x to along z
  omega = state["omega"].to(torch.float32).to(f64)
  ww, (X, Y), mm = len(omega), eps.shape[1:], case["modes"]
  fwd = lambda a, d: torch.roll(a, -1, d) - a
  bwd = lambda a, d: a - torch.roll(a, 1, d)
  e = eps[None, :, :, :, None]
  om = omega[:, None, None, None]

  def apply(v, shift):
    u0, u1 = v[:, 0], v[:, 1]
    b = (-bwd(u0, 2) + bwd(u1, 1)) / e[:, 2]
    c = fwd(u0, 1) + fwd(u1, 2)
    s = shift[:, None, None, None]
    return torch.stack([(om ** 2 * e[:, 1] - s) * u0 - fwd(b, 2) * e[:, 1] + bwd(c, 1),
                        (om ** 2 * e[:, 0] - s) * u1 + fwd(b, 1) * e[:, 0] + bwd(c, 2)], dim=1)

  def iterate(v, shift, n):
    y = apply(v, shift)
    for _ in range(n):
      g = y.reshape(ww, -1, y.shape[-1])
      l = torch.linalg.cholesky(g.transpose(1, 2).contiguous() @ g)
      v = torch.linalg.solve_triangular(l.transpose(1, 2), g, upper=True, left=False)
      v = v.reshape(y.shape)
      y = apply(v, shift)
    w = torch.sum(v * y, dim=(1, 2, 3))
    order = torch.flip(torch.argsort(w, dim=-1), dims=(-1,))
    return (torch.take_along_dim(w, order, -1),
            torch.take_along_dim(v, order[:, None, None, None, :], -1))

  # mode()'s own start vectors: seeded normal numbers.
  start = lambda k: torch.randn((ww, 2, X, Y, k), generator=torch.Generator().manual_seed(0)).to(
      eps.device, f64)
  shift = iterate(start(1), torch.zeros_like(omega), 10)[0]
  w, v = iterate(start(mm), shift[:, 0], case["iters"])
  beta = torch.sqrt(w + shift)
  bz = beta[:, None, None, :]
  hz = (fwd(v[:, 0], 1) + fwd(v[:, 1], 2)) / (1j * bz)
  # E = curl H / (i omega eps) with d/dz = -i beta, backward differences.
  ex = (bwd(hz, 2) + 1j * bz * v[:, 1]) / (1j * om * e[:, 0])
  ey = (-1j * bz * v[:, 0] - bwd(hz, 1)) / (1j * om * e[:, 1])
  power = torch.real(torch.sum(ex * v[:, 1] - ey * v[:, 0], dim=(1, 2)))
  v = v / torch.sqrt(power)[:, None, None, None, :]
  return beta, torch.flip(v, dims=(1,))[:, :, None], None


def _exact_design(case, state):
  f64 = torch.float64
  u = state["u"].detach().to(f64).requires_grad_(True)
  pos = state["pos"].detach().to(f64).requires_grad_(True)
  m, Z, radius = case["m"], case["zz"], case["radius"]
  alpha, c, eta, lo, hi = 0.5, 1.0, 0.5, 0.25, 0.75
  dev = u.device

  def edge(a, n):
    """n more rows and columns on each side, the border's values again."""
    i = torch.clamp(torch.arange(-n, a.shape[0] + n, device=dev), 0, a.shape[0] - 1)
    j = torch.clamp(torch.arange(-n, a.shape[1] + n, device=dev), 0, a.shape[1] - 1)
    return a[i][:, j]

  r = math.ceil(radius - 0.5)
  q = torch.arange(-r, r + 1, dtype=f64) ** 2
  cone = torch.clamp(radius - torch.sqrt(q[:, None] + q[None, :]), min=0)
  cone = (cone / cone.sum()).tolist()
  padded, uf = edge(u, r), 0.0
  for i in range(2 * r + 1):
    for j in range(2 * r + 1):
      if cone[i][j]:
        uf = uf + cone[i][j] * padded[i:i + u.shape[0], j:j + u.shape[1]]
  s = edge((uf >= eta).to(torch.int8), 1)
  mid = s[1:-1, 1:-1]
  rim = ((mid != s[:-2, 1:-1]) | (mid != s[2:, 1:-1]) | (mid != s[1:-1, :-2]) |
         (mid != s[1:-1, 2:]))
  up = torch.where(rim, uf, (torch.sign(uf - eta) + 1) / 2)
  p = edge(uf, 1)
  weight = torch.exp(-c * ((p[2:, 1:-1] - p[:-2, 1:-1]) ** 2 + (p[1:-1, 2:] - p[1:-1, :-2]) ** 2))
  loss = weight * (up * torch.clamp(uf - hi, max=0) ** 2 +
                   (1 - up) * torch.clamp(lo - uf, max=0) ** 2)
  dens = alpha * up + (1 - alpha) * uf
  layers = _layers(dens)
  k = torch.arange(Z, dtype=f64, device=dev)
  inf = torch.full((1,), math.inf, dtype=f64, device=dev)
  low, high = torch.cat([-inf, pos])[:, None], torch.cat([pos, inf])[:, None]
  comps = []
  for comp in range(3):
    v = layers
    if comp != 0:  # half a cell along x, the first sub-pixels repeated
      v = torch.cat([v[:, :1].expand(-1, m, -1), v[:, :-m]], dim=1)
    if comp != 1:
      v = torch.cat([v[:, :, :1].expand(-1, -1, m), v[:, :, :-m]], dim=2)
    tiles = v.reshape(3, case["xx"], 2 * m, case["yy"], 2 * m)
    slope = 12 * (2 * m) * (torch.arange(2 * m, dtype=f64, device=dev) - (m - 0.5)) / (2 * m) ** 2
    gx = torch.mean(tiles * slope[:, None, None], dim=(2, 4))
    gy = torch.mean(tiles * slope, dim=(2, 4))
    avg, inv = torch.mean(tiles, dim=(2, 4)), torch.mean(1 / tiles, dim=(2, 4))
    gs = k + (0.0 if comp == 2 else -0.5)
    ge = gs + 1
    a = torch.minimum(torch.maximum(low, gs), ge)
    b = torch.minimum(torch.maximum(high, gs), ge)
    share = b - a
    mix = lambda f, g: torch.tensordot(f, g, dims=([0], [0]))
    grads = [mix(gx, share), mix(gy, share), mix(avg, share * ((a + b) / 2 - (gs + ge) / 2)) * 12]
    total = sum(g ** 2 for g in grads)
    part = grads[comp] ** 2 / torch.where(total == 0, torch.ones_like(total), total)
    comps.append(1 / (part * mix(inv, share) + (1 - part) / mix(avg, share)))
  eps = torch.stack(comps)
  gu, gp = torch.autograd.grad([eps, loss], [u, pos],
                               [state["g_eps"].to(f64), state["g_loss"].to(f64)])
  return dens.detach(), loss.detach(), eps.detach(), gu, gp


def exact(case, seed):
  state = prepare(case, seed)
  kind = case["kind"]
  if kind == "forward":
    return _Exact(state["calls"][0]).forward()[0]
  if kind == "batch":
    return [_Exact(kw).forward()[0] for kw in state["calls"]]
  if kind in ("gradient", "batch_gradient"):
    got = [_Exact(kw).gradient(lambda out, m=m: _objective(out, m, state["weight"]))
           for kw, m in zip(state["calls"], state["monitors"])]
    if kind == "gradient":
      return got[0]
    return [sum(loss for _, loss, _ in got)] + [grad for _, _, grad in got]
  if kind == "field":
    return _exact_glue(state, state["mode"], state["pos"])
  if kind == "scatter":
    return _exact_scatter(state)
  if kind == "mode":
    return _exact_mode(case, state)
  return _exact_design(case, state)
