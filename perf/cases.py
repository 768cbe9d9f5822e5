"""The work that programs built on qasmhd_amd have it do, as timed cases.

A program holds its domains as device-resident solvers (capi.Solver, a
capi.Batch of them, or a solver behind torch_adjoint.ideal_steps), hands
initial states over as device arrays, runs steps and takes the states back.
Each case is a dict of plain values; ``prepare`` builds what the program
keeps, ``run`` is one pass: initial state in, some steps, final state (and dt
history, gradients) out.  ``exact`` computes the same outputs with plain torch
in float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from qasmhd_amd import capi, torch_adjoint

NG = 4
DEV = "cuda"
F8 = torch.float64
ROE, HLLD, LHLLD, MLAU = 0, 1, 2, 3
FP64, MIXED, FMA64 = 0, 1, 2


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def _case(kind, nx, ny=1, nz=1, steps=4, rmn=HLLD, odr=4, r_k=3, ctw=1, precision=FP64, walls="periodic"):
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, steps=steps, rmn=rmn, odr=odr, r_k=r_k, ctw=ctw,
                precision=precision, walls=walls)


def listed():
    cases = []

    def add(name, c):
        cases.append(dict(c, name=name))

    # the 1D Brio-Wu shock tube of the first tutorial run; latency only
    add("shock1d_1024", _case("shock1d", 1024, steps=32))
    # a small 2D vortex run (64^2), the size of a quick test of a set-up: one
    # round of workgroups or less per launch
    add("turb2d_64", _case("turb2d", 64, 64, steps=8))
    # one member of a parameter study (the sizes of the batched workload)
    add("turb2d_256", _case("turb2d", 256, 256, steps=8))
    # the headline workload: 1024^2 decaying turbulence, FP64 HLLD / WCNS-4
    add("turb2d_1024", _case("turb2d", 1024, 1024, steps=4))
    # a grid that no tile divides, walls on both axes, the Roe solver and the
    # third-order reconstruction with RK2: the options of older set-ups
    add("walls2d_517x389", _case("turb2d", 517, 389, steps=4, rmn=ROE, odr=3, r_k=2, walls="openmirror"))
    # low-Mach shear layer with the all-speed solver at the size it is run at,
    # FP32 reconstruction and fluxes
    add("khi2d_2048_mixed", _case("khi2d", 2048, 2048, steps=2, rmn=MLAU, precision=MIXED))
    # Rayleigh-Taylor with gravity, tall domain with open ends, LHLLD
    add("rt2d_192x1536", _case("rt2d", 192, 1536, steps=4, rmn=LHLLD, walls="open_y"))
    # reconnection with the visco-resistive sub-steps (second order, walls)
    add("mrx2d_1536x192", _case("mrx2d", 1536, 192, steps=4, rmn=LHLLD, odr=2, walls="mirror_y"))
    # 3D turbulence in FP64
    add("turb3d_128", _case("turb3d", 128, 128, 128, steps=2))
    # 3D turbulence in mixed precision, a size that is no multiple of a tile
    add("turb3d_200_mixed", _case("turb3d", 200, 200, 200, steps=2, precision=MIXED))
    # a parameter study: 24 uneven domains advanced together
    add("batch2d_24", dict(_case("batch2d", 0, steps=8), count=24, smallest=128, largest=512))
    # gradient of a loss on the final density with respect to the initial
    # state, 256^2: forward with checkpoints and the discrete adjoint
    add("grad2d_256", dict(_case("grad2d", 256, 256, steps=4), keep=False))
    return cases


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["shock1d", "turb2d", "turb2d", "turb2d", "mixed2d", "rt2d", "mrx2d", "turb3d", "mixed3d",
                       "batch2d", "grad2d"])
    steps = rng.choice([2, 3, 4])
    if kind == "shock1d":
        return _case("shock1d", _log_int(rng, 64, 16384), steps=rng.choice([8, 16, 32]),
                     rmn=rng.choice([ROE, HLLD, LHLLD, MLAU]), odr=rng.choice([2, 3, 4]))
    if kind == "turb2d":
        return _case("turb2d", _log_int(rng, 32, 1024), _log_int(rng, 32, 1024), steps=steps,
                     rmn=rng.choice([HLLD, HLLD, ROE, LHLLD, MLAU]), odr=rng.choice([4, 4, 4, 3, 2]),
                     r_k=rng.choice([3, 3, 2]), ctw=rng.choice([1, 1, 0]), precision=rng.choice([FP64, FP64, FP64, FMA64]),
                     walls=rng.choice(["periodic", "periodic", "openmirror"]))
    if kind == "mixed2d":
        n = _log_int(rng, 128, 2048)
        return _case("khi2d", n, n, steps=2, rmn=rng.choice([MLAU, MLAU, LHLLD]), precision=MIXED)
    if kind == "rt2d":
        nx = _log_int(rng, 32, 256)
        return _case("rt2d", nx, 8 * nx, steps=steps, rmn=LHLLD, walls="open_y")
    if kind == "mrx2d":
        ny = _log_int(rng, 32, 256)
        return _case("mrx2d", 8 * ny, ny, steps=steps, rmn=LHLLD, odr=2, walls="mirror_y")
    if kind in ("turb3d", "mixed3d"):
        mixed = kind == "mixed3d"
        top = 200 if mixed else 144
        return _case("turb3d", _log_int(rng, 24, top), _log_int(rng, 24, top), _log_int(rng, 24, top), steps=2,
                     rmn=rng.choice([HLLD, HLLD, MLAU]), precision=MIXED if mixed else FP64)
    if kind == "batch2d":
        return dict(_case("batch2d", 0, steps=rng.choice([4, 6, 8])), count=rng.randint(4, 24),
                    smallest=rng.randint(64, 160), largest=rng.randint(200, 512))
    return dict(_case("grad2d", _log_int(rng, 48, 288), _log_int(rng, 48, 288), steps=rng.choice([2, 3, 4]),
                      rmn=rng.choice([HLLD, HLLD, MLAU])), keep=rng.choice([False, False, True]))


def _batch_sizes(case):
    """Sizes of the domains of a batch: uneven, from smallest to largest in
    equal ratios, in an order that mixes them."""
    k = case["count"]
    r = math.log(case["largest"] / case["smallest"])
    s = [int(round(case["smallest"] * math.exp(r * i / max(k - 1, 1)))) for i in range(k)]
    return [s[(7 * i) % k] if math.gcd(7, k) == 1 else s[i] for i in range(k)]


# --------------------------------------------------------------------------
# boundary flags and spacing
# --------------------------------------------------------------------------
def _flags(case):
    dn = np.zeros((3, 8), dtype=int)
    if case["kind"] == "shock1d":
        dn[0, :] = 2
    elif case["walls"] == "openmirror":   # open in x, reflecting walls in y
        dn[0, :] = 2
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
    elif case["walls"] == "open_y":
        dn[1, :] = 2
    elif case["walls"] == "mirror_y":
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
    return dn


def _stag():
    st = np.zeros((3, 8), dtype=int)
    st[0, 4] = st[1, 5] = st[2, 6] = 1
    return st


def _gamma(case):
    return 2.0 if case["kind"] == "shock1d" else 5.0 / 3.0


def _interior(case):
    """Interior cells, slowest axis first."""
    if case["kind"] == "shock1d":
        return (case["nx"],)
    if case["kind"] == "turb3d":
        return (case["nz"], case["ny"], case["nx"])
    return (case["ny"], case["nx"])


def _spacing(case):
    """(dx, dy, dz); cells are about square in every case."""
    if case["kind"] == "shock1d":
        return (1.0 / case["nx"], 1.0, 1.0)
    if case["kind"] == "khi2d":
        return (1.0 / case["nx"], 1.0 / case["ny"], 1.0)
    if case["kind"] == "rt2d":
        return (20.0 / case["nx"], 20.0 / case["nx"], 1.0)
    if case["kind"] == "mrx2d":
        return (64.0 / case["nx"], 64.0 / case["nx"], 1.0)
    d = 2.0 * math.pi / max(case["nx"], case["ny"], case["nz"])
    return (d, d, d)


# --------------------------------------------------------------------------
# initial states (float64, on the GPU; a function of the case and the seed)
# --------------------------------------------------------------------------
def _energy(ro, v, b, pr, gam):
    return pr / (gam - 1) + 0.5 * (ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + b[0] ** 2 + b[1] ** 2 + b[2] ** 2)


def _coords(case):
    """Cell-centre coordinates with ghosts, broadcastable, by axis (x, y, z)."""
    dims, d = _interior(case), _spacing(case)
    nd = len(dims)
    out = []
    for a in range(nd):
        n = dims[nd - 1 - a]
        x = (torch.arange(n + 2 * NG, dtype=F8, device=DEV) - NG + 0.5) * d[a]
        out.append(x.reshape([-1 if k == nd - 1 - a else 1 for k in range(nd)]))
    return out


def _modes(rng, case, x, nmodes=6):
    """A smooth periodic field: a sum of random low Fourier modes, about 1 rms."""
    dims, d = _interior(case), _spacing(case)
    nd = len(dims)
    f = 0.0
    for _ in range(nmodes):
        arg = rng.uniform(0, 2 * math.pi)
        for a in range(nd):
            length = dims[nd - 1 - a] * d[a]
            arg = arg + x[a] * (int(rng.integers(-3, 4)) * 2 * math.pi / length)
        f = f + rng.uniform(0.3, 1.0) * torch.cos(arg + torch.zeros([n + 2 * NG for n in dims], dtype=F8, device=DEV))
    return f / math.sqrt(nmodes / 4.0)


def _turbulence(case, seed, mach):
    gam = _gamma(case)
    rng = np.random.default_rng(seed)
    x = _coords(case)
    d = _spacing(case)
    nd = len(x)
    ro = 1.0 + 0.1 * _modes(rng, case, x)
    pr = (1.0 + 0.1 * _modes(rng, case, x)) / gam
    v = [mach * _modes(rng, case, x) for _ in range(3)]
    # face B from a vector potential, so that its discrete divergence is zero
    half = 0.5 * d[0]
    pot = {}
    for a in range(3):
        shifted = [x[c] - (0.0 if c == a else half) for c in range(nd)]
        pot[a] = 0.3 * _modes(rng, case, shifted) if (nd == 3 or a == 2) else None
    sd = lambda f, a: (27.0 * (_sh(f, a, 1) - f) - (_sh(f, a, 2) - _sh(f, a, -1))) / (24.0 * d[a])
    if nd == 3:
        b = [sd(pot[2], 1) - sd(pot[1], 2), sd(pot[0], 2) - sd(pot[2], 0), sd(pot[1], 0) - sd(pot[0], 1) + 0.3]
    else:
        b = [sd(pot[2], 1), -sd(pot[2], 0), 0.3 + 0.1 * _modes(rng, case, x)]
    c = [0.5 * (b[a] + _sh(b[a], a, 1)) if a < nd else b[a] for a in range(3)]
    return torch.stack([ro, ro * v[0], ro * v[1], ro * v[2], b[0], b[1], b[2], _energy(ro, v, c, pr, gam)])


def _initial(case, seed):
    """(state, extras): the state with ghosts filled, and phi / nu / eta / dcmax."""
    kind, gam = case["kind"], _gamma(case)
    rng = np.random.default_rng(1000 + seed)
    extras = {}
    if kind in ("turb2d", "turb3d"):
        u = _turbulence(case, seed, 0.7)
    elif kind == "grad2d":
        u = _turbulence(case, seed, 0.3)
    else:
        x = _coords(case)
        d = _spacing(case)
        full = [n + 2 * NG for n in _interior(case)]
        zero = torch.zeros(full, dtype=F8, device=DEV)
        if kind == "shock1d":
            left = x[0] < rng.uniform(0.4, 0.6)
            jump = rng.uniform(0.9, 1.1)
            ro = torch.where(left, 1.0 * jump + zero, 0.125 + zero)
            pr = torch.where(left, 1.0 * jump + zero, 0.1 + zero)
            v = [zero, zero, zero]
            b = [0.75 + zero, torch.where(left, 1.0 + zero, -1.0 + zero), zero]
            c = b
        elif kind == "khi2d":
            mach, width = 0.01, 0.02
            s = x[1] - 0.5
            vx = 0.5 * mach * (torch.tanh(s / width) - torch.tanh((s - 0.5) / width) - torch.tanh((s + 0.5) / width))
            noise = torch.zeros(full, dtype=F8, device=DEV)
            gen = torch.Generator(device=DEV).manual_seed(seed)
            noise[NG:-NG, NG:-NG] = 2.0 * torch.rand(_interior(case), generator=gen, dtype=F8, device=DEV) - 1.0
            vy = torch.where(torch.abs(s) < 0.05, 1e-3 * mach * noise, zero)
            ro, pr = 1.0 + zero, 1.0 / gam + zero
            v, b = [vx + zero, vy, zero], [0.05 + zero, zero, zero]
            c = b
        elif kind == "rt2d":
            ny = case["ny"]
            y = x[1] - 0.5 * ny * d[1]
            ly, lam, lg = ny * d[1], 1.0, 8 * d[1]
            s0 = 0.35 * ly
            ro = 0.1 + 0.45 * (2.0 + torch.tanh((y - s0) / lam) - torch.tanh((y + s0) / lam)) + zero
            phi = lg * torch.log(torch.cosh(y / lg)) + zero
            # hydrostatic balance from the bottom up
            dp = -0.5 * (ro[1:] + ro[:-1]) * (phi[1:] - phi[:-1])
            pr = 500.0 + torch.cat([zero[:1], torch.cumsum(dp, 0)])
            amp = 0.01 * rng.uniform(0.5, 1.5)
            wave = torch.cos(2 * math.pi * x[0] / 20.0 + rng.uniform(0, 2 * math.pi))
            vy = amp * wave * (torch.exp(-((y - s0) ** 2) / 4) - torch.exp(-((y + s0) ** 2) / 4))
            v, b = [zero, vy, zero], [zero, zero, 1.0 + zero]
            c = b
            extras["phi"] = phi
        else:  # mrx2d: Harris sheet, localised viscosity and resistivity
            xx = x[0] - 0.5 * case["nx"] * d[0]
            yy = x[1] - 0.5 * case["ny"] * d[1]
            b1 = 0.05 * rng.uniform(0.5, 1.5)
            ro = 1.0 / torch.cosh(yy) ** 2 + 0.2 + zero
            bx0 = torch.tanh(yy) + zero
            pr = 0.5 * (1.2 - bx0 * bx0)
            xm, ym = xx - 0.5 * d[0], yy - 0.5 * d[1]
            bump = torch.exp(-(xx * xx + yy * yy) / 4)
            b = [bx0 - b1 * yy * torch.exp(-(xm * xm + yy * yy) / 4), b1 * xx * torch.exp(-(xx * xx + ym * ym) / 4) + zero,
                 zero]
            c = [bx0 - b1 * yy * bump, b1 * xx * bump, zero]
            v = [zero, zero, zero]
            r = torch.sqrt(xx * xx + yy * yy)
            extras["nu"] = 5e-3 * torch.exp(-r)
            extras["eta"] = 5e-3 * torch.exp(-r)
            extras["dcmax"] = float(torch.maximum(2 * extras["nu"], extras["eta"]).max())
        en = _energy(ro, v, c, pr, gam)
        if "phi" in extras:
            en = en + ro * extras["phi"]
        u = torch.stack([ro, ro * v[0], ro * v[1], ro * v[2], b[0], b[1], b[2], en])
    return _bound(u, _flags(case), _stag(), extras.get("phi"), gam).contiguous(), extras


def _members(case, seed):
    """The domains of a batch as cases of their own."""
    for i, n in enumerate(_batch_sizes(case)):
        yield dict(_case("turb2d", n, n, steps=case["steps"], rmn=case["rmn"], odr=case["odr"], r_k=case["r_k"]),
                   name=str(i)), 100 * seed + i


# --------------------------------------------------------------------------
# prepare, run, work
# --------------------------------------------------------------------------
def _solver(case, extras):
    dx, dy, dz = _spacing(case)
    s = capi.Solver([n + 2 * NG for n in _interior(case)], dx, dy, dz, gam=_gamma(case), rmn=case["rmn"],
                    odr=case["odr"], r_k=case["r_k"], ctw=case["ctw"], dn=_flags(case), precision=case["precision"])
    if "phi" in extras:
        s.set_gravity(extras["phi"].cpu().numpy())
    if "nu" in extras:
        s.set_dissipation(extras["nu"].cpu().numpy(), extras["eta"].cpu().numpy(), extras["dcmax"])
    return s


def prepare(case, seed):
    if case["kind"] == "batch2d":
        u0, solvers = [], []
        for c, sd in _members(case, seed):
            u, ex = _initial(c, sd)
            u0.append(u)
            solvers.append(_solver(c, ex))
            solvers[-1].upload_device(u.data_ptr())  # a batch is made of domains that hold a state
            solvers[-1].sync()
        return dict(case=case, u0=u0, solvers=solvers, batch=capi.Batch(solvers), out=[torch.empty_like(u) for u in u0])
    u, ex = _initial(case, seed)
    s = _solver(case, ex)
    if case["kind"] == "grad2d":
        s.adj_keep_stages(case["keep"])
        dts = [_grad_dt(case)] * case["steps"]
        return dict(case=case, u0=u, solver=s, dts=dts, target=_target(case, seed))
    return dict(case=case, u0=u, solver=s, out=torch.empty_like(u))


def _grad_dt(case):
    return 0.15 * _spacing(case)[0]


def _target(case, seed):
    return 1.0 + 0.05 * _modes(np.random.default_rng(7000 + seed), case, _coords(case))


def run(state):
    case = state["case"]
    if case["kind"] == "batch2d":
        for s, u in zip(state["solvers"], state["u0"]):
            s.upload_device(u.data_ptr())
            s.reset_counter()
        hist, _ = state["batch"].run(case["steps"])
        for s, o in zip(state["solvers"], state["out"]):
            s.download_device(o.data_ptr())
        for s in state["solvers"]:
            s.sync()
        return {"states": state["out"], "dt": hist}
    if case["kind"] == "grad2d":
        u = state["u0"].detach().requires_grad_(True)
        final = torch_adjoint.ideal_steps(u, state["solver"], state["dts"])
        loss = ((final[0] - state["target"]) ** 2).sum()
        loss.backward()
        return {"final": final.detach(), "grad": u.grad}
    s = state["solver"]
    s.upload_device(state["u0"].data_ptr())
    s.reset_counter()
    hist, _ = s.run(case["steps"])
    s.download_device(state["out"].data_ptr())
    s.sync()
    return {"state": state["out"], "dt": hist}


def work(case):
    """Compulsory traffic and arithmetic of one pass.  A Runge-Kutta stage is
    a global exchange: it reads the 8 state arrays (and, after the first
    stage, the step's base) and writes 8.  Flops count + - * / sqrt as 1: the
    reconstruction of a cell and the flux of a face per axis, the 4th-order
    differences, the edge EMFs and the face-B update."""
    if case["kind"] == "batch2d":
        per = [work(c) for c, _ in _members(case, 0)]
        return {k: sum(p[k] for p in per) for k in ("bytes", "flops")}
    zones = math.prod(_interior(case))
    nd = len(_interior(case))
    stages = case["steps"] * case["r_k"]
    byts = 8 * 8 * zones * (3 * stages - case["steps"])
    point = {ROE: 610, HLLD: 272, LHLLD: 304, MLAU: 393}[case["rmn"]]
    recon = {1: 160, 2: 300, 3: 480, 4: 859}[case["odr"]]
    edges = {1: 0, 2: 1, 3: 3}[nd]
    flops = zones * stages * (nd * (recon + 44 + point + 36) + edges * 130 + 60)
    if case["kind"] == "mrx2d":   # the dissipative stages, one sub-step a step
        byts *= 2
        flops += zones * stages * 130
    if case["kind"] == "grad2d":  # the adjoint: about twice the forward's arithmetic and state traffic
        byts *= 3
        flops *= 3
    return {"bytes": byts, "flops": flops}


# --------------------------------------------------------------------------
# the scheme in plain torch, float64 (axis 0 = x is the last tensor axis)
# --------------------------------------------------------------------------
def _sh(f, a, k):
    """f at index + k along axis a (wraps at the array's end, where no cell
    that is kept reads)."""
    return torch.roll(f, -k, dims=f.dim() - 1 - a)


def _map_ghosts(f, a, st, dn):
    n = f.shape[f.dim() - 1 - a]
    src, fac = list(range(n)), [1.0] * n
    if dn == 0:
        for i in range(NG):
            src[i], src[n - 1 - i] = n - 2 * NG + i, 2 * NG - 1 - i
    elif abs(dn) == 1:
        for i in range(NG):
            src[i], fac[i] = 2 * NG - 1 + st - i, float(dn)
        for i in range(NG - st):
            src[n - 1 - i], fac[n - 1 - i] = n - 2 * NG + st + i, float(dn)
    else:
        for i in range(NG):
            src[i], fac[i] = NG, 0.25 * (2 + dn)
        for i in range(NG - st):
            src[n - 1 - i], fac[n - 1 - i] = n - 1 - NG + st, 0.25 * (2 + dn)
    dim = f.dim() - 1 - a
    g = f.index_select(dim, torch.tensor(src, device=f.device))
    if min(fac) != 1.0:
        g = g * torch.tensor(fac, dtype=F8, device=f.device).reshape([-1 if k == dim else 1 for k in range(f.dim())])
    return g


def _bc(f, st, dn):
    for a in range(f.dim()):
        f = _map_ghosts(f, a, int(st[a]), int(dn[a]))
    return f


def _bound(u, dn, st, phi=None, gam=None):
    out = [_bc(u[m], st[:, m], dn[:, m]) for m in range(8)]
    if phi is not None:  # hydrostatic energy in the y ghosts
        fac = (2.0 - gam) / (gam - 1.0)
        ro, en = out[0], out[7].clone()
        n = en.shape[0]
        for rows, b in ((slice(0, NG), NG), (slice(n - NG, n), n - NG - 1)):
            en[rows] = en[b] - fac * ro[b] * (phi[rows] - phi[b])
        out[7] = en
    return torch.stack(out)


def _sqrt(x):
    """sqrt with derivative zero at zero."""
    pos = x > 0
    return torch.where(pos, torch.sqrt(torch.where(pos, x, torch.ones_like(x))), torch.zeros_like(x))


def _div(p, q, ok):
    """p / q where ok, else 0 (no infinities in the branch not taken)."""
    return torch.where(ok, p / torch.where(ok, q, torch.ones_like(q)), torch.zeros_like(p))


def _linear(odr, f):
    if odr == 1:
        return f[2], f[2]
    if odr == 2:
        return (-f[1] + 5 * f[2] + 2 * f[3]) / 6, (-f[3] + 5 * f[2] + 2 * f[1]) / 6
    if odr == 3:
        return 0.125 * (-f[1] + 6 * f[2] + 3 * f[3]), 0.125 * (-f[3] + 6 * f[2] + 3 * f[1])
    side = lambda a, b, c, d, e: 0.003125 * (9 * a - 56 * b + 234 * c + 144 * d - 11 * e)
    return side(*f), side(*f[::-1])


def _nonlinear(odr, f):
    """Left state at i+1/2 and right state at i-1/2 from f = i-2 .. i+2."""
    if odr == 1:
        return f[2], f[2]
    if odr == 2:
        a, b = f[2] - f[1], f[3] - f[2]
        zero = torch.zeros_like(a)
        d = 0.5 * (torch.minimum(torch.maximum(a, b), zero) + torch.maximum(torch.minimum(a, b), zero))
        return f[2] + d, f[2] - d
    if odr == 3:
        t = (f[3] - 2 * f[2] + f[1]) ** 2
        s0, s1 = 1 + t / ((f[1] - f[2]) ** 2 + 1e-40), 1 + t / ((f[3] - f[2]) ** 2 + 1e-40)

        def side(a, b, up, dn):
            w = 0.25 * a / (0.25 * a + 0.75 * b)
            return 0.5 * (w * (-up + 3 * f[2]) + (1 - w) * (f[2] + dn))
        return side(s0, s1, f[1], f[3]), side(s1, s0, f[3], f[1])

    def smooth(a, b):
        return 1.0 / (((13.0 / 12.0) * b * b + 0.25 * a * a) ** 2 + 1e-40)
    s0 = smooth(f[0] - 4 * f[1] + 3 * f[2], f[0] - 2 * f[1] + f[2])
    s1 = smooth(f[1] - f[3], f[1] - 2 * f[2] + f[3])
    s2 = smooth(f[4] - 4 * f[3] + 3 * f[2], f[4] - 2 * f[3] + f[2])

    def side(s0, s2, g):
        w0, w1, w2 = 0.075 * s0, 0.650 * s1, 0.275 * s2
        den = w0 + w1 + w2
        w0, w1 = w0 / den, w1 / den
        return 0.125 * (w0 * (3 * g[0] - 10 * g[1] + 15 * g[2]) + w1 * (-g[1] + 6 * g[2] + 3 * g[3])
                        + (1 - w0 - w1) * (3 * g[2] + 6 * g[3] - g[4]))
    return side(s0, s2, f), side(s2, s0, f[::-1])


def _centre(odr, f, a):
    """Face values (at i-1/2) to cell centres along axis a."""
    if odr <= 2:
        return 0.5 * (f + _sh(f, a, 1))
    return 0.0625 * (9.0 * (f + _sh(f, a, 1)) - (_sh(f, a, -1) + _sh(f, a, 2)))


def _diff(odr, f, a):
    if odr <= 2:
        return _sh(f, a, 1) - f
    return (27.0 * (_sh(f, a, 1) - f) - (_sh(f, a, 2) - _sh(f, a, -1))) / 24.0


def _face_states(odr, q, a, bn, gam):
    """Characteristic reconstruction along axis a of q = (ro, vn, vt, vu, bt,
    bu, pr): states at i-1/2 (left from the cell below, right of this cell)."""
    s = [[_sh(f, a, m) for m in range(-2, 3)] for f in q]
    ro0, bt0, bu0, pr0 = q[0], q[4], q[5], q[6]
    fast = ro0 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) > gam * pr0
    cs2, ca2, ct2 = gam * pr0 / ro0, bn * bn / ro0, (bt0 ** 2 + bu0 ** 2) / ro0
    cb2 = cs2 + ca2 + ct2
    cf2 = 0.5 * (cb2 + _sqrt(torch.abs(cb2 * cb2 - 4 * cs2 * ca2)))
    rcf, sro = ro0 * _sqrt(cf2), _sqrt(ro0)
    w = [[] for _ in range(7)]
    for m in range(5):
        r, vn, vt, vu, bt, bu, p = (s[k][m] for k in range(7))
        ptot = bt0 * bt + bu0 * bu + p
        w[0].append(torch.where(fast, -rcf * vn + ptot, vn))
        w[1].append(cf2 * r - ptot)
        w[2].append(torch.where(fast, rcf * vn + ptot, ptot))
        w[3].append(sro * vt + bt)
        w[4].append(sro * vt - bt)
        w[5].append(sro * vu + bu)
        w[6].append(sro * vu - bu)
    pairs = [_nonlinear(odr, f) for f in w]
    out = []
    for side in range(2):
        c = [p[side] for p in pairs]
        mag = -0.5 * bt0 * (c[3] - c[4]) - 0.5 * bu0 * (c[5] - c[6])
        v = [torch.where(fast, (0.5 * c[0] + c[1] + 0.5 * c[2]) / cf2, (c[1] + c[2]) / cf2),
             torch.where(fast, 0.5 * (c[2] - c[0]) / rcf, c[0]),
             0.5 * (c[3] + c[4]) / sro, 0.5 * (c[5] + c[6]) / sro, 0.5 * (c[3] - c[4]), 0.5 * (c[5] - c[6]),
             torch.where(fast, 0.5 * (c[0] + c[2]), c[2]) + mag]
        for k in range(1, 6):
            still = torch.ones_like(fast)
            for m in range(5):
                still = still & (s[k][m] == 0)
            v[k] = torch.where(still, torch.zeros_like(v[k]), v[k])
        bad = (v[0] <= 1e-12) | (v[6] <= 1e-12)
        for k in (0, 1, 6):
            v[k] = torch.where(bad, q[k], v[k])
        out.append(v)
    return [_sh(f, a, -1) for f in out[0]], out[1]


def _flux(rmn, L, R, bn, gam, dv0, dv1):
    if rmn == ROE:
        return _flux_roe(L, R, bn, gam)
    return (_flux_mlau if rmn == MLAU else _flux_hlld)(L, R, bn, gam, dv0, dv1, rmn == LHLLD)


def _side(q, bn, gam):
    ro, vn, vt, vu, bt, bu, pr = q
    pm = 0.5 * (bt * bt + bu * bu)
    v2 = vn * vn + vt * vt + vu * vu
    en = pr / (gam - 1) + pm + 0.5 * ro * v2
    ca2 = bn * bn / ro

    def speed2(c2):
        cb2 = c2 + ca2 + 2 * pm / ro
        return 0.5 * (cb2 + _sqrt(torch.abs(cb2 * cb2 - 4 * c2 * ca2)))
    return pr + pm, en, speed2(gam * pr / ro), speed2(v2)


def _flux_hlld(L, R, bn, gam, dv0, dv1, low):
    one, zero = torch.ones_like(bn), torch.zeros_like(bn)
    sgn = torch.where(bn > 0, one, -one)
    (ptl, enl, cfl2, ccl2), (ptr, enr, cfr2, ccr2) = _side(L, bn, gam), _side(R, bn, gam)
    cmax = _sqrt(torch.maximum(cfl2, cfr2))
    sl = torch.minimum(zero, torch.minimum(L[1], R[1]) - cmax)
    sr = torch.maximum(zero, torch.maximum(L[1], R[1]) + cmax)
    ml, mr = L[0] * (sl - L[1]), R[0] * (sr - R[1])
    jump = 1.0
    theta = 1.0
    if low:
        theta = torch.minimum(one, (cmax - torch.minimum(dv0, zero)) / (cmax - torch.minimum(dv1, zero))) ** 4
        mcc = torch.minimum(one, _sqrt(torch.maximum(ccl2, ccr2)) / cmax)
        jump = mcc * (2 - mcc)
    vc = (mr * R[1] - ml * L[1] - theta * (ptr - ptl)) / (mr - ml)
    pc = (mr * ptl - ml * ptr + jump * mr * ml * (R[1] - L[1])) / (mr - ml)

    def star(q, s, m, pt, en):
        sv, sc = s - q[1], s - vc
        ro2 = m / sc
        rh = m * sc - bn * bn
        ok = torch.abs(rh) > 1e-8
        dv = _div((q[1] - vc) * bn, rh, ok)
        fb = torch.where(ok, _div(m * sv - bn * bn, rh, ok), one)
        vt, vu, bt, bu = q[2] + dv * q[4], q[3] + dv * q[5], fb * q[4], fb * q[5]
        en2 = (sv * en - pt * q[1] + pc * vc + bn * (q[2] * q[4] + q[3] * q[5] - vt * bt - vu * bu)) / sc
        return ro2, vt, vu, bt, bu, en2
    ro2l, vtl, vul, btl, bul, e2l = star(L, sl, ml, ptl, enl)
    ro2r, vtr, vur, btr, bur, e2r = star(R, sr, mr, ptr, enr)
    a, b = _sqrt(ro2l), _sqrt(ro2r)
    vt3 = (b * vtr + a * vtl + (btr - btl) * sgn) / (a + b)
    vu3 = (b * vur + a * vul + (bur - bul) * sgn) / (a + b)
    bt3 = (a * btr + b * btl + a * b * (vtr - vtl) * sgn) / (a + b)
    bu3 = (a * bur + b * bul + a * b * (vur - vul) * sgn) / (a + b)
    vb3 = vt3 * bt3 + vu3 * bu3
    e3l = e2l - a * (vtl * btl + vul * bul - vb3) * sgn
    e3r = e2r + b * (vtr * btr + vur * bur - vb3) * sgn
    left = vc > 0
    in2l = vc - torch.abs(bn) / a > 0
    in2r = ~(vc + torch.abs(bn) / b > 0)
    pick = lambda l, m, r: torch.where(in2l, l, torch.where(in2r, r, m))
    ro = torch.where(left, ro2l, ro2r)
    vt, vu, bt, bu = pick(vtl, vt3, vtr), pick(vul, vu3, vur), pick(btl, bt3, btr), pick(bul, bu3, bur)
    en = pick(e2l, torch.where(left, e3l, e3r), e2r)
    return [ro * vc, ro * vc * vc + pc - 0.5 * bn * bn, ro * vt * vc - bn * bt, ro * vu * vc - bn * bu,
            bt * vc - bn * vt, bu * vc - bn * vu, (en + pc) * vc - bn * (vt * bt + vu * bu)]


def _flux_mlau(L, R, bn, gam, dv0, dv1, low):
    one, zero = torch.ones_like(bn), torch.zeros_like(bn)
    sgn = torch.where(bn > 0, one, -one)
    bna, bn2 = torch.abs(bn), bn * bn
    (ptl, enl, cfl2, ccl2), (ptr, enr, cfr2, ccr2) = _side(L, bn, gam), _side(R, bn, gam)
    rol, ror, vnl, vnr = L[0], R[0], L[1], R[1]
    cf = _sqrt(torch.maximum(cfl2, cfr2))
    sl = torch.minimum(zero, torch.minimum(vnl, vnr) - cf)
    sr = torch.maximum(zero, torch.maximum(vnl, vnr) + cf)
    theta = torch.minimum(one, (cf - torch.minimum(dv0, zero)) / (cf - torch.minimum(dv1, zero))) ** 4

    def split(m, e):  # e = +1 left, -1 right
        sn = torch.where(m > 0, one, -one)
        m2 = m * m - 1
        b0 = 0.5 * (1 + e * sn)
        b1 = 0.25 * (m + e) ** 2 * (2 - e * m) + e * 0.1875 * m * m2 * m2
        f1 = e * (0.25 * (m + e) ** 2 + 0.125 * m2 * m2)
        sup = sn * m > 1
        return torch.where(sup, b0, b1), torch.where(sup, b0 * m, f1)
    bfl, ffl = split(vnl / cf, 1.0)
    bfr, ffr = split(vnr / cf, -1.0)
    mn = ffl + ffr
    mf = mn * cf - torch.maximum(1 - torch.abs(mn), zero) * theta / cf * (ptr - ptl) / (rol + ror)
    up = mf > 0
    pick = lambda l, r: torch.where(up, l, r)
    mf = mf * pick(rol, ror)
    mfl, mfr = pick(mf, zero), pick(zero, mf)
    cm = _sqrt(torch.maximum(ccl2, ccr2))
    pt = (bfl * ptl + bfr * ptr - 0.25 * bfl * bfr * (rol + ror) * cm * (vnr - vnl)
          - 0.5 * (1 - cm / cf) * (bfl + bfr - 1) * (ptl + ptr))
    sc = pick(sl, sr)
    vden = mf + pick(rol * (sl - vnl), ror * (sr - vnr))
    ok = (torch.abs(vden) > 1e-8) & (sc != 0)
    vc = torch.where(ok, _div(mf * sc, vden, ok), pick(vnl, vnr))

    def star(q, s):
        slv, slc = s - q[1], s - vc
        rh = q[0] * slv * slc - bn2
        ok = torch.abs(rh) > 1e-8
        k = _div(vc - q[1], rh, ok)
        dvt, dvu, dbt, dbu = -bn * q[4] * k, -bn * q[5] * k, bn2 * q[4] * k / slc, bn2 * q[5] * k / slc
        cmp = slv / slc
        return (_sqrt(q[0] * cmp), dvt, dvu, dbt, dbu, dvt + q[2], dvu + q[3], dbt + q[4] * cmp, dbu + q[5] * cmp)
    al, dvtl, dvul, dbtl, dbul, vt2l, vu2l, bt2l, bu2l = star(L, sl)
    ar, dvtr, dvur, dbtr, dbur, vt2r, vu2r, bt2r, bu2r = star(R, sr)
    clip = lambda x: sgn * torch.minimum(torch.maximum(zero, x), bna)
    fl, fr = al / (al + ar), ar / (al + ar)
    blb, brb = clip(fl * (bna + ar * vc)), clip(fr * (bna - al * vc))
    blv, brv = clip(fr * (bna + mf / ar)), clip(fl * (bna - mf / al))
    rv = torch.maximum(bna - pick(one, -one) * vc * pick(al, ar), zero)
    cb = rv / (al + ar)
    cv = al * ar * cb
    bnvt = blb * vt2l + brb * vt2r + cb * (bt2r - bt2l) - vc * pick(dbtl, dbtr)
    bnvu = blb * vu2l + brb * vu2r + cb * (bu2r - bu2l) - vc * pick(dbul, dbur)
    bnbt = blv * bt2l + brv * bt2r + cv * (vt2r - vt2l) - mf * pick(dvtl, dvtr)
    bnbu = blv * bu2l + brv * bu2r + cv * (vu2r - vu2l) - mf * pick(dvul, dvur)
    fmt, fmu = mfl * L[2] + mfr * R[2] - bnbt, mfl * L[3] + mfr * R[3] - bnbu
    fbt, fbu = mfl * L[4] / rol + mfr * R[4] / ror - bnvt, mfl * L[5] / rol + mfr * R[5] / ror - bnvu
    vb1 = pick(L[2] * L[4] + L[3] * L[5], R[2] * R[4] + R[3] * R[5])
    vb2 = pick(vt2l * bt2l + vu2l * bu2l, vt2r * bt2r + vu2r * bu2r)
    rv2 = (mf * vc - bn2) ** 2
    vb3 = _div((fmt * vc + fbt * bn) * (fmt * bn + fbt * mf) + (fmu * vc + fbu * bn) * (fmu * bn + fbu * mf), rv2,
               rv2 > 1e-16)
    bnvb = sgn * (bna * (sc * vb2 - vc * vb1) / pick(sl - vc, sr - vc) + rv * (vb3 - vb2))
    return [mf, mfl * vnl + mfr * vnr + pt - 0.5 * bn2, fmt, fmu, fbt, fbu,
            mfl * (enl + ptl) / rol + mfr * (enr + ptr) / ror - bnvb]


def _flux_roe(L, R, bn, gam):
    one, zero = torch.ones_like(bn), torch.zeros_like(bn)
    g1, g2 = gam - 1, gam - 2
    a, b = _sqrt(L[0]), _sqrt(R[0])
    ro = a * b
    avg = lambda l, r: (a * l + b * r) / (a + b)
    vn, vt, vu = avg(L[1], R[1]), avg(L[2], R[2]), avg(L[3], R[3])
    bt, bu = avg(R[4], L[4]), avg(R[5], L[5])
    enth = lambda q: (gam / g1 * q[6] + bn * bn + q[4] ** 2 + q[5] ** 2) / q[0] + 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)
    hl, hr = enth(L), enth(R)
    h = avg(hl, hr)
    sgn = torch.where(bn > 0, one, -one)
    dbt, dbu = R[4] - L[4], R[5] - L[5]
    db2 = 0.5 * g2 / g1 * (dbt ** 2 + dbu ** 2) / (a + b) ** 2
    v2 = 0.5 * (vn * vn + vt * vt + vu * vu)
    bb = bn * bn + bt * bt + bu * bu
    c2, a2 = g1 * (h - v2 - db2 - bb / ro), g1 * (h - v2 - db2) - g2 * bb / ro
    ca2, cb2 = bn * bn / ro, (bt * bt + bu * bu) / ro
    cf2 = 0.5 * (a2 + _sqrt(cb2 * (a2 + c2 + ca2) + (c2 - ca2) ** 2))
    cs2 = c2 * ca2 / cf2
    cf, cs, ca, c = _sqrt(cf2), _sqrt(cs2), _sqrt(ca2), _sqrt(c2)
    perp = bt * bt + bu * bu
    has = perp - 1e-8 > 0
    norm = _sqrt(torch.where(has, perp, perp + 1))
    et, eu = torch.where(has, bt / norm, math.sqrt(0.5) * one), torch.where(has, bu / norm, math.sqrt(0.5) * one)
    reg = perp / ro + torch.abs(ca2 - c2) - 1e-8 > 0
    den = _sqrt(torch.maximum(zero, cf2 - cs2) + torch.where(reg, zero, one))
    alf = torch.where(reg, _sqrt(torch.maximum(zero, cf2 - ca2)) / den, one)
    als = torch.where(reg, _sqrt(torch.maximum(zero, cf2 - c2)) / den, zero)
    t1 = et * dbt + eu * dbu
    t2 = (R[6] - L[6] + 0.5 * ((L[4] + R[4]) * dbt + (L[5] + R[5]) * dbu) + g2 * (bt * dbt + bu * dbu)) / g1
    t3 = eu * dbt - et * dbu
    s1, mt, mu = ro * (R[1] - L[1]), ro * (R[2] - L[2]), ro * (R[3] - L[3])
    s2, s3 = et * mt + eu * mu, eu * mt - et * mu
    rr = _sqrt(ro)
    p11, p12 = als * cf / rr, -alf * c2 / cf / rr
    p21, p22 = alf * (cf2 - c2 * g2 / g1), als * (cs2 - c2 * g2 / g1)
    q11, q12, q21, q22 = alf * cf, als * cs, -als * ca * sgn, alf * c * sgn
    dp, dq = p11 * p22 - p12 * p21, q11 * q22 - q12 * q21
    wf, ws = (p22 * t1 - p12 * t2) / dp, (-p21 * t1 + p11 * t2) / dp
    xf, xs = (q22 * s1 - q12 * s2) / dq, (-q21 * s1 + q11 * s2) / dq
    w = {"pf": 0.5 * (wf + xf), "mf": 0.5 * (wf - xf), "ps": 0.5 * (ws + xs), "ms": 0.5 * (ws - xs),
         "pa": 0.5 * (rr * t3 - sgn * s3), "ma": 0.5 * (rr * t3 + sgn * s3)}
    w["e"] = (R[0] - L[0]) - alf * (w["pf"] + w["mf"]) - als * (w["ps"] + w["ms"])
    lam = {"pf": vn + cf, "mf": vn - cf, "ps": vn + cs, "ms": vn - cs, "pa": vn + ca, "ma": vn - ca, "e": vn}
    bv = et * vt + eu * vu
    vec = {}
    for k, e in (("pf", 1.0), ("mf", -1.0)):
        vec[k] = [alf, alf * (vn + e * cf), alf * vt - e * als * et * ca * sgn, alf * vu - e * als * eu * ca * sgn,
                  als * et * cf / rr, als * eu * cf / rr,
                  alf * (v2 + db2 + e * cf * vn + cf2 / g1 + (cf2 - c2) * g2 / g1) - e * als * ca * bv * sgn]
    for k, e in (("ps", 1.0), ("ms", -1.0)):
        vec[k] = [als, als * (vn + e * cs), als * vt + e * c * sgn * alf * et, als * vu + e * c * sgn * alf * eu,
                  -c2 * alf * et / cf / rr, -c2 * alf * eu / cf / rr,
                  als * (v2 + db2 + e * cs * vn + cs2 / g1 + (cs2 - c2) * g2 / g1) + e * alf * c * bv * sgn]
    for k, e in (("pa", 1.0), ("ma", -1.0)):
        vec[k] = [zero, zero, -e * sgn * eu, e * sgn * et, eu / rr, -et / rr, -e * (eu * vt - et * vu) * sgn]
    vec["e"] = [one, vn, vt, vu, zero, zero, v2 + db2]

    def phys(q, hh):
        m = q[0] * q[1]
        return [m, m * q[1] + q[6] + 0.5 * (q[4] ** 2 + q[5] ** 2 - bn * bn), m * q[2] - bn * q[4], m * q[3] - bn * q[5],
                q[1] * q[4] - q[2] * bn, q[1] * q[5] - q[3] * bn, m * hh - bn * (bn * q[1] + q[4] * q[2] + q[5] * q[3])]
    fl, fr = phys(L, hl), phys(R, hr)
    return [0.5 * (fl[i] + fr[i] - sum(torch.abs(lam[k]) * w[k] * vec[k][i] for k in w)) for i in range(7)]


def _cuct(ro, va, vb, ba, bb, a, b):
    """Upwind weight of the edge shared by four cells in the plane (a, b)."""
    four = lambda f: 0.25 * (f + _sh(f, a, -1) + _sh(f, b, -1) + _sh(_sh(f, a, -1), b, -1))
    rc = 1.0 / _sqrt(four(ro))
    x = torch.abs(four(va)) + torch.abs(0.5 * (ba + _sh(ba, b, -1)) * rc)
    y = torch.abs(four(vb)) + torch.abs(0.5 * (bb + _sh(bb, a, -1)) * rc)
    return (x + 0.5e-12) / (x + y + 1e-12)


def _edge(odr, f, a):
    lo, hi = _linear(odr, [_sh(f, a, m) for m in range(-2, 3)])
    return _sh(lo, a, -1) + hi


def _box(shape, extra=None):
    """Mask of the interior, with one more face at the upper end of an axis."""
    m = torch.ones(shape, dtype=torch.bool, device=DEV)
    nd = len(shape)
    for a in range(nd):
        n = shape[nd - 1 - a]
        keep = torch.zeros(n, dtype=torch.bool, device=DEV)
        keep[NG:n - NG + (1 if a == extra else 0)] = True
        m = m & keep.reshape([-1 if k == nd - 1 - a else 1 for k in range(nd)])
    return m


_RK = {1: [(0.0, 1.0)], 2: [(0.0, 1.0), (0.5, 0.5)], 3: [(0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)]}


def _step(u, dt, case, dn, st, d, phi=None):
    """One Runge-Kutta step of the ideal equations, u with its ghosts filled."""
    odr, rmn, gam = case["odr"], case["rmn"], _gamma(case)
    nd = u.dim() - 1
    inside = _box(u.shape[1:])
    base = u
    for ca, cb in _RK[case["r_k"]]:
        ro, b = u[0], [u[4], u[5], u[6]]
        v = [u[1] / ro, u[2] / ro, u[3] / ro]
        c = [_bc(_centre(odr, b[a], a), (0, 0, 0), dn[:, 4 + a]) if (a < nd and nd > 1) else b[a] for a in range(3)]
        en = u[7] if phi is None else u[7] - ro * phi
        pr = (gam - 1) * (en - 0.5 * (ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + c[0] ** 2 + c[1] ** 2 + c[2] ** 2))
        dv = []
        for a in range(nd):
            f = torch.minimum(_sh(v[a], a, 1) - v[a], v[a] - _sh(v[a], a, -1))
            dv.append(_bc(f, (0, 0, 0), [-dn[k, 1 + a] if k == a else dn[k, 1 + a] for k in range(3)]))
        div = {m: 0.0 for m in (0, 1, 2, 3, 4, 5, 6, 7)}
        emf = [0.0, 0.0, 0.0]
        for a in range(nd):
            t, w = (a + 1) % 3, (a + 2) % 3
            L, R = _face_states(odr, [ro, v[a], v[t], v[w], c[t], c[w], pr], a, c[a], gam)
            dv0 = v[a] - _sh(v[a], a, -1)
            others = [torch.minimum(_sh(dv[k], a, -1), dv[k]) for k in (t, w) if k < nd]
            dv1 = torch.minimum(others[0], others[1]) if len(others) == 2 else (others[0] if others else torch.zeros_like(ro))
            F = _flux(rmn, L, R, b[a], gam, dv0, dv1)
            fe = F[6] if phi is None else F[6] + F[0] * 0.5 * (_sh(phi, a, -1) + phi)
            flux = {0: F[0], 1 + a: F[1], 1 + t: F[2], 1 + w: F[3], 7: fe}
            for k, fk in ((t, F[4]), (w, F[5])):
                if k >= nd:
                    flux[4 + k] = fk      # no edges along this axis: an ordinary flux
                elif nd > 1:
                    # central part b_k v_n - b_n v_k, and the rest of the flux, to the edge along the third axis
                    lo0, hi0 = _linear(odr, [_sh(c[k] * v[a], a, m) for m in range(-2, 3)])
                    lo1, hi1 = _linear(odr, [_sh(v[k], a, m) for m in range(-2, 3)])
                    fc = 0.5 * (_sh(lo0 - _sh(b[a], a, 1) * lo1, a, -1) + hi0 - b[a] * hi1)
                    e = 3 - a - k
                    pa, pb = (e + 1) % 3, (e + 2) % 3
                    ct = _cuct(ro, v[pa], v[pb], b[pa], b[pb], pa, pb) if case["ctw"] else 0.5
                    sgn, wt = (-0.5, 1.0 - ct) if k == t else (0.5, ct)
                    emf[e] = emf[e] + sgn * (_edge(odr, fk - fc, k) + wt * _edge(odr, fc, k))
            for m, f in flux.items():
                div[m] = div[m] - dt / d[a] * _diff(odr, f, a)
        new = [u[m] for m in range(8)]
        for m in (0, 1, 2, 3, 7) + tuple(4 + a for a in range(nd, 3)) + ((5, 6) if nd == 1 else ()):
            new[m] = torch.where(inside, ca * base[m] + cb * (u[m] + div[m]), u[m])
        if phi is not None:
            for a in (0, 1):
                force = -cb * new[0] * 0.5 * (_sh(phi, a, 1) - _sh(phi, a, -1)) * dt / d[a]
                new[1 + a] = torch.where(inside, new[1 + a] + force, new[1 + a])
        if nd > 1:
            for a in range(nd):
                t, w = (a + 1) % 3, (a + 2) % 3
                db = 0.0
                if t < nd:
                    db = db - dt / d[t] * _diff(odr, emf[w], t)
                if w < nd:
                    db = db + dt / d[w] * _diff(odr, emf[t], w)
                new[4 + a] = torch.where(_box(u.shape[1:], a), ca * base[4 + a] + cb * (b[a] + db), b[a])
        u = _bound(torch.stack(new), dn, st, phi, gam)
    return u


def _dissipate(u, dt, case, dn, st, d, nu, eta):
    """One Runge-Kutta step of the viscous and resistive terms (2D)."""
    odr = case["odr"]
    inside = _box(u.shape[1:])
    base = u
    c4 = lambda f, a: _centre(odr, _sh(f, a, -1), a)   # cell centres to the face at i-1/2
    d4 = lambda f, a: _diff(odr, _sh(f, a, -1), a)
    for ca, cb in _RK[case["r_k"]]:
        ro, b = u[0], [u[4], u[5], u[6]]
        v = [u[1] / ro, u[2] / ro, u[3] / ro]
        grad = lambda f, a: d4(f, a) / d[a]
        ex = 0.5 * (eta + _sh(eta, 1, -1)) * grad(b[2], 1)   # eta j at the edges
        ey = -0.5 * (eta + _sh(eta, 0, -1)) * grad(b[2], 0)
        e4 = 0.25 * (eta + _sh(eta, 0, -1) + _sh(eta, 1, -1) + _sh(_sh(eta, 0, -1), 1, -1))
        ez = e4 * (grad(b[1], 0) - grad(b[0], 1))
        div = {m: 0.0 for m in (0, 1, 2, 3, 6, 7)}
        rnu = ro * nu
        for a in (0, 1):
            o = 1 - a
            mu = 0.5 * (_sh(rnu, a, -1) + rnu)
            cross = lambda f: c4(0.5 * (_sh(f, o, 1) - _sh(f, o, -1)), a) / d[o]
            tau = {a: -mu * (4.0 / 3.0 * grad(v[a], a) - 2.0 / 3.0 * cross(v[o])),
                   o: -mu * (grad(v[o], a) + cross(v[a])), 2: -mu * grad(v[2], a)}
            fen = sum(tau[k] * c4(v[k], a) for k in (0, 1, 2))
            # resistive fluxes: -E x B along the axis, E and B averaged to the face
            ezf = 0.5 * (ez + _sh(ez, o, 1))
            bo = c4(0.5 * (b[o] + _sh(b[o], o, 1)), a)
            bz = c4(b[2], a)
            if a == 0:
                fen, fbz = fen + ey * bz - ezf * bo, ey
            else:
                fen, fbz = fen + ezf * bo - ex * bz, -ex
            for m, f in ((1, tau[0]), (2, tau[1]), (3, tau[2]), (6, fbz), (7, fen)):
                div[m] = div[m] - dt / d[a] * _diff(odr, f, a)
        new = [u[m] for m in range(8)]
        for m in (0, 1, 2, 3, 6, 7):
            new[m] = torch.where(inside, ca * base[m] + cb * (u[m] + div[m]), u[m])
        new[4] = torch.where(_box(u.shape[1:], 0), ca * base[4] + cb * (u[4] - dt / d[1] * _diff(odr, ez, 1)), u[4])
        new[5] = torch.where(_box(u.shape[1:], 1), ca * base[5] + cb * (u[5] + dt / d[0] * _diff(odr, ez, 0)), u[5])
        u = _bound(torch.stack(new), dn, st)
    return u


def _cfl(u, case, dn, d, phi=None):
    gam, nd = _gamma(case), u.dim() - 1
    ro = u[0]
    c = [0.5 * (u[4 + a] + _sh(u[4 + a], a, 1)) if (a < nd and nd > 1) else u[4 + a] for a in range(3)]
    v = [u[1] / ro, u[2] / ro, u[3] / ro]
    b2 = c[0] ** 2 + c[1] ** 2 + c[2] ** 2
    en = u[7] if phi is None else u[7] - ro * phi
    pr = (gam - 1) * (en - 0.5 * (ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + b2))
    s = torch.sqrt(sum(v[a] ** 2 for a in range(nd))) + torch.sqrt((gam * pr + b2) / ro)
    vmax = max(1.0, float(s[tuple([slice(NG, -NG)] * nd)].max()))
    return 0.4 * min(d[:nd]) / vmax


def _run_exact(case, seed):
    u, ex = _initial(case, seed)
    dn, st, d, phi = _flags(case), _stag(), _spacing(case), ex.get("phi")
    dt = _cfl(u, case, dn, d, phi)
    hist = []
    for n in range(1, case["steps"] + 1):
        hist.append(dt)
        u = _step(_bound(u, dn, st, phi, _gamma(case)), dt, case, dn, st, d, phi)
        if "nu" in ex:
            nc = 1 + int(2 * (ex["dcmax"] * dt) / min(d[0], d[1]) ** 2)
            for _ in range(nc):
                u = _dissipate(_bound(u, dn, st), dt / nc, case, dn, st, d, ex["nu"], ex["eta"])
        if n % 2 == 0:
            dt = _cfl(u, case, dn, d, phi)
    return u, np.array(hist)


def exact(case, seed):
    """What run returns for these inputs, from the equations above."""
    if case["kind"] == "batch2d":
        done = [_run_exact(c, sd) for c, sd in _members(case, seed)]
        return {"states": [u for u, _ in done], "dt": np.stack([h for _, h in done])}
    if case["kind"] == "grad2d":
        u0, _ = _initial(case, seed)
        u0 = u0.requires_grad_(True)
        dn, st, d = _flags(case), _stag(), _spacing(case)
        u = _bound(u0, dn, st)
        for _ in range(case["steps"]):
            u = _step(u, _grad_dt(case), case, dn, st, d)
        ((u[0] - _target(case, seed)) ** 2).sum().backward()
        return {"final": u.detach(), "grad": u0.grad}
    u, hist = _run_exact(case, seed)
    return {"state": u, "dt": hist}
