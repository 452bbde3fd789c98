"""The work that programs give this library, as cases that can be timed and checked.

A case is a dict of plain values; `listed()` gives the standing ones, `draw(rng)`
one more of the same ranges.  `prepare(case, seed)` builds what a program has in
hand before the call (a scheduler, its history, sample points), `run(state)` makes
the call through the package's public entry points and returns its results,
`work(case)` counts what the call cannot do without, and `exact(case, seed)`
gives the results in plain torch / numpy double precision where that is quick.

Kinds of case:
  hostloop1d  one step of a driver that keeps the history on the host: rho down,
              Poisson and fit on host buffers, the new slice up
  run1d       a whole 1D run to T, energies and coefficient history back
  sweep1d     many independent 1D runs stepped together, energies back
  adjoint1d   J = time-integrated field energy and its gradient with respect to
              the initial condition, forward and backward, as an optimiser calls it
  diag1d      a driver's output step: metrics row, field and f on plotting grids,
              phase flow
  step3d      one device-resident 3D time step from a stored history (an isolated
              step, or step n of a run)
  metrics3d   the metrics row of a 3D output step

The histories that steps and diagnostics start from are written in closed form:
damped (or, for two-stream, growing and saturating) standing waves of the family's
wave number, as the linear phase of such runs has, with amplitudes and phases from
the seed.  In 3D the potential is a sum of one wave per axis.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import config as nconf
from numericalflowiteration_amd.adjoint import time_integrated_energy

FLOP_1D, FLOP_3D = 30.0, 475.0      # per characteristic step, order 4 (FMA = 2)


def listed():
    return [
        # the smallest call: one early step of a small linear run driven from the host,
        # where launches, copies and waits are the whole cost
        dict(name="hostloop1d_landau_64x256_n32", kind="hostloop1d", family="landau", Nx=64, Nu=256, n=32,
             precision="fp64"),
        # linear Landau damping to T = 30: 481 short steps, bound by latency
        dict(name="run1d_landau_64x256_t30", kind="run1d", family="landau", Nx=64, Nu=256, T=30.0, dt=0.0625,
             precision="fp64"),
        # a grid chosen by eye, no power of two on either axis
        dict(name="run1d_landau_100x515_t20", kind="run1d", family="landau", Nx=100, Nu=515, T=20.0, dt=0.0625,
             precision="fp64"),
        # two-stream instability to T = 50 at production resolution, both forms of the trace
        dict(name="run1d_twostream_256x1024_t50", kind="run1d", family="twostream", Nx=256, Nu=1024, T=50.0, dt=0.03125,
             precision="fp64"),
        dict(name="run1d_twostream_256x1024_t50_fp32c", kind="run1d", family="twostream", Nx=256, Nu=1024, T=50.0,
             dt=0.03125, precision="fp32c"),
        # a parameter study: 512 runs of uneven grids and initial conditions, one device
        dict(name="sweep1d_512_t20_fp32c", kind="sweep1d", runs=512, T=20.0, precision="fp32c"),
        # gradient of the time-integrated energy with respect to eight mode amplitudes
        dict(name="adjoint1d_multimode_128x512_t20", kind="adjoint1d", family="multimode", Nx=128, Nu=512, T=20.0,
             dt=0.0625, precision="fp64"),
        # an output step of the 1D driver in mid run
        dict(name="diag1d_twostream_256x1024_n400", kind="diag1d", family="twostream", Nx=256, Nu=1024, n=400, points=512,
             precision="fp64"),
        # the mean step of the 3D Landau run (16^3 x 32^3, T = 20), both forms of the trace
        dict(name="step3d_landau_16_32_n80", kind="step3d", family="landau", Nx=16, Ny=16, Nz=16, Nu=32, Nv=32, Nw=32,
             n=80, precision="fp64"),
        dict(name="step3d_landau_16_32_n80_fp32c", kind="step3d", family="landau", Nx=16, Ny=16, Nz=16, Nu=32, Nv=32,
             Nw=32, n=80, precision="fp32c"),
        # a larger, uneven 3D grid early in a run (more points than one workgroup solves)
        dict(name="step3d_bump_20x18x20_n24", kind="step3d", family="bump", Nx=20, Ny=18, Nz=20, Nu=22, Nv=18, Nw=20,
             n=24, precision="fp64"),
        # the metrics row of a 3D output step
        dict(name="metrics3d_landau_16_16_n40", kind="metrics3d", family="landau", Nx=16, Ny=16, Nz=16, Nu=16, Nv=16,
             Nw=16, n=40, precision="fp64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hostloop1d", "run1d", "run1d", "sweep1d", "adjoint1d", "diag1d", "step3d", "step3d", "step3d",
                       "metrics3d"])
    precision = rng.choice(["fp64", "fp64", "fp32c"])
    if kind in ("step3d", "metrics3d"):
        c = dict(kind=kind, family=rng.choice(["landau", "twostream", "bump"]), precision=precision)
        even = rng.random() < 0.4
        N = [rng.choice([8, 16])] * 3 if even else [rng.randint(8, 20) for _ in range(3)]
        V = [rng.choice([12, 16, 24])] * 3 if even else [rng.randint(9, 24) for _ in range(3)]
        nodes = N[0] * N[1] * N[2] * V[0] * V[1] * V[2]
        budget = 2.5e9 if kind == "step3d" else 6e8
        n = max(2, min(_log(rng, 6, 90), int(budget / nodes)))
        c.update(zip(("Nx", "Ny", "Nz"), N), **dict(zip(("Nu", "Nv", "Nw"), V)), n=n)
        return c
    if kind == "sweep1d":
        return dict(kind=kind, runs=_log(rng, 6, 160), T=rng.randint(6, 40) / 4.0, precision=precision)
    Nx = rng.choice([32, 64, 128, 256]) if rng.random() < 0.5 else _log(rng, 24, 400)
    Nu = max(16, min(1100, int(Nx * rng.uniform(2.0, 5.0))))
    family = rng.choice(["landau", "twostream", "multimode"])
    c = dict(kind=kind, family=family, Nx=Nx, Nu=Nu, precision=precision)
    if kind == "hostloop1d":
        c.update(n=_log(rng, 4, 400))
    elif kind == "run1d":
        c.update(T=rng.randint(10, 40) / 2.0, dt=rng.choice([0.0625, 0.05, 0.1]))
    elif kind == "adjoint1d":
        c.update(Nx=min(Nx, 160), Nu=min(Nu, 520), T=rng.randint(4, 24) / 2.0, dt=0.0625)
    else:
        c.update(n=_log(rng, 8, 500), points=_log(rng, 48, 600), precision="fp64")
    return c


# ---- configurations and seeded inputs -------------------------------------------

_K1 = {"landau": 0.5, "twostream": 0.2, "multimode": 0.5}
_V1 = {"landau": 10.0, "twostream": 8.0, "multimode": 10.0}
_F1 = {"landau": nconf.F0_LANDAU_1D, "twostream": nconf.F0_TWOSTREAM_1D, "multimode": nconf.F0_MULTIMODE_1D}
_K3 = {"landau": 0.5, "twostream": 0.5, "bump": 0.3}
_V3 = {"landau": 6.0, "twostream": 8.0, "bump": 9.0}
_F3 = {"landau": nconf.F0_LANDAU_3D, "twostream": nconf.F0_TWOSTREAM_3D, "bump": nconf.F0_BUMPONTAIL_3D}


def _precision(case):
    return nufi.FP32C if case["precision"] == "fp32c" else nufi.FP64


def _alpha(case, r):
    base = {"landau": 0.01, "twostream": 0.001, "multimode": 0.0, "bump": 0.03}[case["family"]]
    return base * r.uniform(0.8, 1.25)


def _config1(case, seed):
    r = np.random.default_rng(seed)
    k, v = _K1[case["family"]], _V1[case["family"]]
    alpha = _alpha(case, r)
    modes = list(0.02 * r.random(8)) if case["family"] == "multimode" else None
    dt = case.get("dt", 0.0625)
    T = case["T"] if "T" in case else dt * (case["n"] + 0.5)
    return nufi.config_1d(case["Nx"], case["Nu"], dt, T, 0.0, 2 * math.pi / k, -v, v, _F1[case["family"]],
                          alpha=alpha, k=k, modes=modes)


def _config3(case, seed):
    r = np.random.default_rng(seed)
    k, v = _K3[case["family"]], _V3[case["family"]]
    return nufi.config_3d((case["Nx"], case["Ny"], case["Nz"]), (case["Nu"], case["Nv"], case["Nw"]), 0.125,
                          0.125 * (case["n"] + 0.5), (0.0, 2 * math.pi / k), (-v, v), _F3[case["family"]],
                          alpha=_alpha(case, r), k=k)


def _wave(case, N, dx, k, alpha, slices, dt, r):
    """Coefficients of one standing wave per slice, (slices, N + 3): amplitude alpha/k^2,
    damped, or growing to a saturated level for two-stream."""
    t = dt * np.arange(slices)
    omega, phase, shift = r.uniform(1.3, 1.5), r.uniform(0, 2 * math.pi), r.uniform(0, 2 * math.pi)
    if case["family"] == "twostream":
        amp = np.minimum(alpha * np.exp(0.25 * t), 0.15) * (1.0 + 0.05 * np.cos(omega * t + phase))
    else:
        amp = alpha * np.exp(-0.15 * t) * np.cos(omega * t + phase)
    out = np.zeros((slices, N + 3))
    i = np.arange(N + 3) % N
    for m, part in ((1, 1.0), (2, 0.2 * r.uniform(0.5, 1.0))):
        km = k * m
        fit = (4.0 + 2.0 * math.cos(km * dx)) / 6.0
        out += (part * amp / km ** 2)[:, None] * (np.cos(km * dx * (i - 1) + shift) / fit)[None, :]
    return out


def _history1(case, seed, conf, slices):
    r = np.random.default_rng(seed + 7919)
    alpha = conf.f0.alpha or 0.02
    return _wave(case, conf.Nx, conf.dx, _K1[case["family"]], alpha, slices, conf.dt, r)


def _history3(case, seed, conf, slices):
    r = np.random.default_rng(seed + 7919)
    k = _K3[case["family"]]
    axes = ((conf.Nx, conf.dx), (conf.Ny, conf.dy), (conf.Nz, conf.dz))
    return [_wave(case, N, d, k, conf.f0.alpha, slices, conf.dt, r) for N, d in axes]


def _outer3(a):
    return a[2][:, :, None, None] + a[1][:, None, :, None] + a[0][:, None, None, :]


def _points(case, seed, conf):
    """The plotting grids of a 1D output step, shifted a little by the seed."""
    r = np.random.default_rng(seed + 104729)
    P = case["points"]
    xs = conf.x_min + conf.Lx * (np.arange(2 * P) + r.random()) / (2 * P)
    gx = conf.x_min + conf.Lx * (np.arange(P) + r.random()) / P
    gv = conf.u_min + (conf.u_max - conf.u_min) * (np.arange(P) + r.random()) / P
    X, V = np.meshgrid(gx, gv)
    return xs, np.ascontiguousarray(X).ravel(), np.ascontiguousarray(V).ravel()


def _sweep_confs(case, seed):
    return [nufi.sweep_config(q, T=case["T"]) for q in nufi.sweep_runs(case["runs"], seed=nconf.SWEEP_SEED + seed)]


# ---- what a program holds, and one pass --------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "sweep1d":
        return dict(kind=kind, batch=nufi.BatchScheduler(_sweep_confs(case, seed), precision=_precision(case)))
    if kind == "adjoint1d":
        conf = _config1(case, seed)
        f = conf.f0
        values = [f.a[i] for i in range(f.n_modes)] if f.kind == nconf.F0_MULTIMODE_1D else [f.alpha]
        return dict(kind=kind, conf=conf, precision=_precision(case), values=torch.tensor(values, dtype=torch.float64))
    if kind == "run1d":
        return dict(kind=kind, sched=nufi.GpuScheduler(_config1(case, seed), precision=_precision(case)))
    n = case["n"]
    conf = _config3(case, seed) if kind in ("step3d", "metrics3d") else _config1(case, seed)
    sched = nufi.GpuScheduler(conf, precision=_precision(case))
    state = dict(kind=kind, sched=sched, n=n)
    slices = n + 1 if kind in ("diag1d", "metrics3d") else n
    if conf.dim == 3:
        hist = _outer3(_history3(case, seed, conf, slices))
    else:
        hist = _history1(case, seed, conf, slices)
    hist = np.ascontiguousarray(hist).ravel()
    if slices:
        sched.upload_history(hist, 0, slices)
    if kind == "hostloop1d":
        state["coeffs"] = np.concatenate([hist, np.zeros(sched.stride_t)])
        state["rho"] = np.zeros(conf.Nx)
    elif kind == "diag1d":
        state["points"] = _points(case, seed, conf)
    sched.synchronize()
    return state


def run(state):
    kind = state["kind"]
    if kind == "sweep1d":
        # a study keeps the energies of every run (growth and damping rates are read off them)
        b = state["batch"]
        b.run()
        b.synchronize()
        return dict(energies=np.concatenate([b.energies(r) for r in range(b.n_runs)]))
    if kind == "adjoint1d":
        a = state["values"].clone().requires_grad_(True)
        J = time_integrated_energy(a, state["conf"], state["precision"])
        J.backward()
        return dict(J=J.detach(), grad=a.grad)
    s = state["sched"]
    if kind == "run1d":
        e = s.run()
        return dict(energies=e, history=s.history())
    n = state["n"]
    if kind == "hostloop1d":
        rho, coeffs, st = state["rho"], state["coeffs"], s.stride_t
        rho[:] = 0.0
        s.compute_rho(n)
        s.download_rho(rho)
        out = dict(rho=rho.copy())
        out["energy"] = s.poisson_solve(rho)
        coeffs[n * st:(n + 1) * st] = s.interpolate(rho)
        s.upload_phi(n, coeffs)
        out["phi"], out["slice"] = rho.copy(), coeffs[n * st:(n + 1) * st].copy()
        return out
    if kind == "step3d":
        return dict(energy=s.step(n), slice=s.history(n, n + 1))
    metrics = np.zeros(4)
    s.compute_metrics(n)
    s.download_metrics(metrics)
    if kind == "metrics3d":
        return dict(metrics=metrics)
    xs, X, V = state["points"]
    E, rho = s.sample_field(n, xs)
    f = s.sample_f(n, X, V)
    xf, vf = s.phase_flow(n, X, V)
    return dict(metrics=metrics, E=E, rho=rho, f=f, x=xf, v=vf)


# ---- what a pass cannot do without -------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "sweep1d":
        confs = _sweep_confs(case, 1)
        cs = sum(c.char_steps(0, c.Nt + 1) for c in confs)
        return dict(bytes=8.0 * sum(c.Nt + 1 for c in confs), flops=FLOP_1D * cs)
    if kind in ("step3d", "metrics3d"):
        conf = _config3(case, 1)
        n = case["n"]
        if kind == "step3d":
            return dict(bytes=8.0 * (n + 1) * conf.stride_t(), flops=FLOP_3D * conf.n_nodes() * n)
        return dict(bytes=8.0 * (n + 1) * conf.stride_t() + 32.0, flops=FLOP_3D * conf.n_nodes() * (n + 1))
    conf = _config1(case, 1)
    st = conf.stride_t()
    if kind == "run1d":
        return dict(bytes=8.0 * (conf.Nt + 1) * (st + 1), flops=FLOP_1D * conf.char_steps(0, conf.Nt + 1))
    if kind == "adjoint1d":
        # the forward run, then a forward and a reverse pass of each step
        return dict(bytes=8.0 * (conf.Nt + 1) * st, flops=3 * FLOP_1D * conf.char_steps(0, conf.Nt + 1))
    n = case["n"]
    if kind == "hostloop1d":
        return dict(bytes=8.0 * ((n + 1) * st + 3 * conf.Nx), flops=FLOP_1D * conf.n_nodes() * n)
    pts = case["points"] ** 2
    return dict(bytes=8.0 * ((n + 1) * st + 6 * pts + 8 * case["points"]),
                flops=FLOP_1D * (n + 1) * (conf.n_nodes() + 2.0 * pts))


# ---- the same results in plain double precision -----------------------------------

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _tensor(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


def _cell_poly(c, N):
    """(3, N): dphi/dt = q0 + q1 t + q2 t^2 in every cell, from coefficients c (.., N + 3)."""
    d = c[..., 1:] - c[..., :-1]
    d0, d1, d2 = d[..., 0:N], d[..., 1:N + 1], d[..., 2:N + 2]
    return torch.stack([(d0 + d1) / 2, d1 - d0, (d0 - 2 * d1 + d2) / 2], dim=-2)


def _foot(hist, n, s, u, conf_dt, dx, N, first_half=False):
    """Backward characteristics of one axis: positions s in cells, velocities u."""
    s, u = s.clone(), u.clone()
    if n == 0:
        return s, u
    cd, q = conf_dt / dx, _cell_poly(hist, N)

    def kick(m, h):
        fl = torch.floor(s)
        t = s - fl
        g = q[m].index_select(1, fl.long().remainder_(N))
        u.add_(torch.addcmul(g[0], t, torch.addcmul(g[1], t, g[2])), alpha=-h * cd / conf_dt)

    if first_half:
        kick(n, conf_dt / 2)
    for m in range(n - 1, -1, -1):
        s.sub_(u, alpha=cd)
        kick(m, conf_dt / 2 if m == 0 else conf_dt)
    return s, u


def _axis_f0(conf, axis):
    """The velocity factor of one axis of the 3D families."""
    kind = conf.f0.kind
    if kind == nconf.F0_TWOSTREAM_3D and axis == 1:
        return lambda v: torch.exp(-(v - 2.4) ** 2 / 2) + torch.exp(-(v + 2.4) ** 2 / 2)
    if kind == nconf.F0_BUMPONTAIL_3D and axis == 0:
        return lambda v: 0.9 * torch.exp(-v * v / 2) + 0.2 * torch.exp(-2 * (v - 4.5) ** 2)
    return lambda v: torch.exp(-v * v / 2)


def _f0_1(conf, x, u):
    f = conf.f0
    if f.kind == nconf.F0_MULTIMODE_1D:
        p = 1.0 + sum(f.a[m] * torch.cos(f.k * (m + 1) * x) for m in range(f.n_modes))
    else:
        p = 1.0 + f.alpha * torch.cos(f.k * x)
    g = torch.exp(-u * u / 2) / math.sqrt(2 * math.pi)
    return p * g * u * u if f.kind == nconf.F0_TWOSTREAM_1D else p * g


def _kappa(N, L):
    i = torch.arange(N, dtype=torch.float64, device=_dev())
    return torch.where(2 * i < N, i, N - i) * (2 * math.pi / L)


def _symbol(N):
    th = 2 * math.pi * torch.arange(N, dtype=torch.float64, device=_dev()) / N
    return (1.0 + 4.0 * torch.exp(1j * th) + torch.exp(2j * th)) / 6.0


def _field(rho, Ls):
    """(phi, coefficients without padding, energy) of a rho of one or three axes (.., y, x)."""
    Ns = list(reversed(rho.shape))
    dims = list(range(rho.dim()))
    k2 = sum((_kappa(N, L) ** 2).reshape([-1] + [1] * a) for a, (N, L) in enumerate(zip(Ns, Ls)))
    sym = 1.0
    for a, N in enumerate(Ns):
        sym = sym * _symbol(N).reshape([-1] + [1] * a)
    F = torch.fft.fftn(rho, dim=dims)
    k2.view(-1)[0] = 1.0
    F.view(-1)[0] = 0.0
    phi = F / k2
    e = math.prod(Ls) / 2 * (F.abs() ** 2 / k2).sum() / rho.numel() ** 2
    return torch.fft.ifftn(phi, dim=dims).real, torch.fft.ifftn(phi / sym, dim=dims).real, e


def _pad(c):
    for a, N in enumerate(c.shape):
        c = c.index_select(a, torch.arange(N + 3, device=c.device) % N)
    return c


def _nodes1(conf):
    ix = torch.arange(conf.Nx, dtype=torch.float64, device=_dev())
    iu = torch.arange(conf.Nu, dtype=torch.float64, device=_dev())
    s = ix[:, None].expand(conf.Nx, conf.Nu).reshape(-1).contiguous()
    u = (conf.u_min + iu * conf.du + conf.du / 2)[None, :].expand(conf.Nx, conf.Nu).reshape(-1).contiguous()
    return s, u


def _rho1(conf, hist, n):
    s, u = _foot(hist, n, *_nodes1(conf), conf.dt, conf.dx, conf.Nx)
    return -conf.du * _f0_1(conf, conf.x_min + s * conf.dx, u).reshape(conf.Nx, conf.Nu).sum(1)


def _metrics(f, v2, w):
    pos = torch.clamp(f, min=1e-300)
    return torch.stack([w * f.sum(), w * (f * f).sum(), w * (v2 * f / 2).sum(), -w * (f * torch.log(pos)).sum()])


def _np(t):
    return t.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "sweep1d":
        return None
    if kind == "run1d":
        conf = _config1(case, seed)
        if conf.Nt * (conf.Nt + 1) // 2 > 130000:
            return None
        hist = torch.zeros(conf.Nt + 1, conf.Nx + 3, dtype=torch.float64, device=_dev())
        en = []
        for n in range(conf.Nt + 1):
            _, c, e = _field(_rho1(conf, hist[:n], n), [conf.Lx])
            hist[n] = _pad(c)
            en.append(e)
        return dict(energies=_np(torch.stack(en)), history=_np(hist).ravel())
    if kind == "adjoint1d":
        return _exact_adjoint(_config1(case, seed))
    n = case["n"]
    if kind in ("hostloop1d", "diag1d"):
        conf = _config1(case, seed)
        hist = _tensor(_history1(case, seed, conf, n + 1 if kind == "diag1d" else n))
        if kind == "hostloop1d":
            rho = _rho1(conf, hist, n)
            phi, c, e = _field(rho, [conf.Lx])
            return dict(rho=_np(rho), energy=float(e), phi=_np(phi), slice=_np(_pad(c)))
        return _exact_diag(case, seed, conf, hist, n)
    conf = _config3(case, seed)
    waves = [_tensor(w) for w in _history3(case, seed, conf, n + 1 if kind == "metrics3d" else n)]
    grid = ((conf.Nx, conf.Nu, conf.u_min, conf.du, conf.x_min, conf.dx),
            (conf.Ny, conf.Nv, conf.v_min, conf.dv, conf.y_min, conf.dy),
            (conf.Nz, conf.Nw, conf.w_min, conf.dw, conf.z_min, conf.dz))
    k, alpha = (0.3, 0.03) if conf.f0.kind == nconf.F0_BUMPONTAIL_3D else (conf.f0.k, conf.f0.alpha)
    const = (2 * math.pi) ** -1.5 * (0.5 if conf.f0.kind == nconf.F0_TWOSTREAM_3D else 1.0)
    # the potential is a sum over the axes, so each axis is traced by itself
    cosx, g, vel = [], [], []
    for a, (N, V, v0, dv, x0, dx) in enumerate(grid):
        s = torch.arange(N, dtype=torch.float64, device=_dev())[:, None].expand(N, V).reshape(-1)
        v = (v0 + torch.arange(V, dtype=torch.float64, device=_dev()) * dv + dv / 2)[None, :].expand(N, V).reshape(-1)
        sf, vf = _foot(waves[a], n, s, v, conf.dt, dx, N, first_half=kind == "metrics3d")
        cosx.append(torch.cos(k * (x0 + sf * dx)).reshape(N, V))
        g.append(_axis_f0(conf, a)(vf).reshape(N, V))
        vel.append(v.reshape(N, V))
    if kind == "step3d":
        m0 = [q.sum(1) for q in g]
        m1 = [(q * c).sum(1) for q, c in zip(g, cosx)]
        def outer(a, b, c):
            return c[:, None, None] * b[None, :, None] * a[None, None, :]
        rho = outer(*m0) + alpha * (outer(m1[0], m0[1], m0[2]) + outer(m0[0], m1[1], m0[2]) + outer(m0[0], m0[1], m1[2]))
        _, c, e = _field(-(conf.du * conf.dv * conf.dw) * const * rho, [conf.Lx, conf.Ly, conf.Lz])
        return dict(energy=float(e), slice=_np(_pad(c)).ravel())
    total = torch.zeros(4, dtype=torch.float64, device=_dev())
    w = conf.du * conf.dv * conf.dw
    for iz in range(conf.Nz):
        def axes(q):      # (y, x, w, v, u)
            return (q[0][None, :, None, None, :], q[1][:, None, None, :, None], q[2][iz][None, None, :, None, None])
        cx, cy, cz = axes(cosx)
        gx, gy, gz = axes(g)
        vx, vy, vz = axes(vel)
        f = const * (gx * gy * gz) * (1.0 + alpha * (cx + cy + cz))
        total += _metrics(f, vx * vx + vy * vy + vz * vz, w)
    return dict(metrics=_np(total))


def _exact_diag(case, seed, conf, hist, n):
    xs, X, V = (_tensor(a) for a in _points(case, seed, conf))
    c = hist[n]
    z = (xs - conf.x_min) / conf.dx
    fl = torch.floor(z)
    t, i = z - fl, fl.long() % conf.Nx
    q = _cell_poly(c, conf.Nx)[:, i]
    E = -(q[0] + t * (q[1] + t * q[2])) / conf.dx
    rho = -(q[1] + 2 * t * q[2]) / conf.dx ** 2
    s, u = _nodes1(conf)
    sf, uf = _foot(hist, n, s, u, conf.dt, conf.dx, conf.Nx, first_half=True)
    m = _metrics(_f0_1(conf, conf.x_min + sf * conf.dx, uf), u * u, conf.du * conf.dx)
    s, v = _foot(hist, n, (X - conf.x_min) / conf.dx, V, conf.dt, conf.dx, conf.Nx, first_half=True)
    x = conf.x_min + s * conf.dx
    f = _f0_1(conf, x, v)
    if n <= 1:
        x, v = X, V
    x = x - conf.Lx * torch.floor(x / conf.Lx)
    return dict(metrics=_np(m), E=_np(E), rho=_np(rho), f=_np(f), x=_np(x), v=_np(v))


def _exact_adjoint(conf):
    """J and its gradient by carrying the tangents of all parameters forward."""
    f0 = conf.f0
    many = f0.kind == nconf.F0_MULTIMODE_1D
    P = f0.n_modes if many else 1
    if conf.Nt * (conf.Nt + 1) // 2 > 60000:
        return None
    N, cd, dt = conf.Nx, conf.dt / conf.dx, conf.dt
    hist = torch.zeros(conf.Nt + 1, P + 1, 3, N, dtype=torch.float64, device=_dev())
    k2 = _kappa(N, conf.Lx) ** 2
    k2[0] = 1.0
    J = torch.zeros(P + 1, dtype=torch.float64, device=_dev())
    s0, u0 = _nodes1(conf)
    for n in range(conf.Nt + 1):
        s = torch.cat([s0[None], torch.zeros(P, s0.numel(), dtype=torch.float64, device=_dev())])
        u = torch.cat([u0[None], torch.zeros(P, s0.numel(), dtype=torch.float64, device=_dev())])
        for m in range(n - 1, -1, -1):
            s.sub_(u, alpha=cd)
            fl = torch.floor(s[0])
            t = s[0] - fl
            g = hist[m].index_select(2, fl.long().remainder_(N))
            p = torch.addcmul(g[:, 0], t, torch.addcmul(g[:, 1], t, g[:, 2]))
            p[1:].addcmul_(torch.addcmul(g[0, 1], t, g[0, 2], value=2.0), s[1:])
            u.add_(p, alpha=-(0.5 if m == 0 else 1.0) / conf.dx * dt)
        x, dx_, v = conf.x_min + s[0] * conf.dx, s[1:] * conf.dx, u[0]
        e = torch.exp(-v * v / 2) / math.sqrt(2 * math.pi)
        amps = [f0.a[m] for m in range(P)] if many else [f0.alpha]
        h, hx, ha = torch.ones_like(x), torch.zeros_like(x), []
        for m, a in enumerate(amps):
            km = f0.k * (m + 1)
            ha.append(torch.cos(km * x))
            h, hx = h + a * ha[m], hx - a * km * torch.sin(km * x)
        ha = torch.stack(ha)
        if f0.kind == nconf.F0_TWOSTREAM_1D:
            G, Gv = e * v * v, e * v * (2.0 - v * v)
        else:
            G, Gv = e, -e * v
        f = torch.cat([(h * G)[None], ha * G + hx * G * dx_ + h * Gv * u[1:]])
        rho = -conf.du * f.reshape(P + 1, conf.Nx, conf.Nu).sum(2)
        F = torch.fft.fft(rho)
        F[:, 0] = 0.0
        w = conf.Lx / 2 / N ** 2 / k2
        J[0] += dt * (w * F[0].abs() ** 2).sum()
        J[1:] += dt * 2 * (w * (F[0].conj() * F[1:]).real).sum(1)
        c = torch.fft.ifft(F / k2 / _symbol(N)).real
        hist[n] = _cell_poly(c.index_select(1, torch.arange(N + 3, device=c.device) % N), N)
    return dict(J=_np(J[0]), grad=_np(J[1:]))
