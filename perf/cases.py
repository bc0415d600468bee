"""Timed cases of the GPU time advance: what a program that integrates
problems with this package has it do, through its public entry points.

A case is one block (or ensemble) of one of six families:

  tgv       3-D periodic Taylor-Green type flow, constant viscosity, any of
            the convective schemes (opensbli_amd/apps/taylor_green.py)
  wave      2-D periodic Euler density wave (apps/euler_wave.py)
  plate     flat plate / shock-wave boundary-layer block: stretched
            wall-normal grid, Sutherland viscosity, inlet, wall, outflow, 2-D
            (apps/katzer_sbli.py, with the sensor) or 3-D (apps/flat_plate.py)
  curv      Euler wave on a general curvilinear grid, 2-D or 3-D
            (apps/euler_wave_curvilinear.py)
  tubes     1-D shock tubes: one block (apps/sod_shock_tube.py), or an
            ensemble of uneven ones in one launch (ensemble.py)
  adjoint   checkpointed 2-D Kelvin-Helmholtz run, forward and backward
            (opensbli_amd/adjoint.py)

One pass sets the state on the device, advances `steps` iterations and
reads the state back (ensembles and gradients likewise).  `exact` restates
the schemes in plain torch, double precision, on arrays padded by their
halos.
"""
import math
import random

import numpy as np
import torch
import torch.utils.checkpoint

from opensbli_amd import adjoint
from opensbli_amd.ensemble import Ensemble, ensemble_parameters, instance_problem
from opensbli_amd.native import Block
from opensbli_amd.problems import (euler_wave_curvilinear, euler_wave_curvilinear_3d, flat_plate, kelvin_helmholtz)

F64 = torch.float64
DEV = "cuda"


def listed():
    return [
        # the Sod app's block: every step is launches and latency
        dict(name="sod_200", family="tubes", count=1, n=200, conv="weno_z", rk="rk3", steps=50),
        # the Taylor-Green script as shipped: 64^3, central skew, low-storage RK
        dict(name="tgv_64_central", family="tgv", nx=64, ny=64, nz=64, conv="central_skew", avg="roe", rk="ls3",
             steps=10),
        # the benchmark's block: WENO5-Z, 256^3
        dict(name="tgv_256_weno_z", family="tgv", nx=256, ny=256, nz=256, conv="weno_z", avg="roe", rk="rk3",
             steps=2),
        # the same block with the central scheme
        dict(name="tgv_256_central", family="tgv", nx=256, ny=256, nz=256, conv="central_skew", avg="roe", rk="ls3",
             steps=3),
        # sizes that fill neither tiles nor waves, the most expensive reconstruction
        dict(name="tgv_ragged_teno6", family="tgv", nx=131, ny=97, nz=75, conv="teno6", avg="roe", rk="rk3", steps=3),
        # 2-D periodic WENO5-JS with simple averaging at the Euler wave app's size
        dict(name="wave_400_weno_js", family="wave", nx=400, ny=400, conv="weno_js", avg="simple", rk="ls3",
             steps=20),
        # the 3-D flat plate of the benchmark
        dict(name="plate_480x256x128", family="plate", nx=480, ny=256, nz=128, conv="weno_z", sensor=False,
             wall="adiabatic_wall", steps=2),
        # the Katzer block: 2-D, adaptive TENO5, isothermal wall
        dict(name="katzer_500x250", family="plate", nx=500, ny=250, nz=0, conv="teno5", sensor=True,
             wall="isothermal_wall", steps=20),
        # general curvilinear grid at the benchmark's size
        dict(name="curv_1024", family="curv", ndim=2, n=1024, conv="weno_z", avg="roe", steps=4),
        # 512 uneven tubes integrated in one launch
        dict(name="ensemble_512", family="tubes", count=512, n=4000, conv="weno_z", rk="rk3", steps=0),
        # gradients of a 2-D run, shock capturing and central viscous
        dict(name="adjoint_512_weno_z", family="adjoint", n=512, conv="weno_z", viscous=False, steps=20, every=10),
        dict(name="adjoint_512_central", family="adjoint", n=512, conv="central_skew", viscous=True, steps=20,
             every=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


CHAR = ["weno_z", "weno_js", "teno5", "teno6"]


def draw(rng):
    family = rng.choice(["tgv", "tgv", "tgv", "wave", "plate", "plate", "curv", "tubes", "tubes", "adjoint"])
    if family == "tgv":
        conv = rng.choice(CHAR + ["central_skew", "central_skew", "central_cons"])
        return dict(family=family, nx=_log(rng, 24, 256), ny=_log(rng, 24, 256), nz=_log(rng, 24, 256), conv=conv,
                    avg=rng.choice(["roe", "simple"]), rk=rng.choice(["rk3", "ls3"]), steps=2)
    if family == "wave":
        return dict(family=family, nx=_log(rng, 32, 1024), ny=_log(rng, 32, 1024),
                    conv=rng.choice(CHAR + ["central_skew"]), avg=rng.choice(["roe", "simple"]),
                    rk=rng.choice(["rk3", "ls3"]), steps=5)
    if family == "plate":
        three = rng.random() < 0.6
        conv, sensor = rng.choice([("weno_z", False), ("weno_z", False), ("teno5", True), ("teno6", False)])
        return dict(family=family, nx=_log(rng, 48, 400 if three else 800), ny=_log(rng, 40, 220 if three else 400),
                    nz=_log(rng, 16, 110) if three else 0, conv=conv, sensor=sensor,
                    wall=rng.choice(["adiabatic_wall", "isothermal_wall"]), steps=2 if three else 8)
    if family == "curv":
        if rng.random() < 0.5:
            return dict(family=family, ndim=2, n=_log(rng, 48, 1024), conv=rng.choice(CHAR),
                        avg=rng.choice(["roe", "simple"]), steps=4)
        return dict(family=family, ndim=3, n=_log(rng, 24, 100), conv=rng.choice(CHAR),
                    avg=rng.choice(["roe", "simple"]), steps=2)
    if family == "tubes":
        if rng.random() < 0.5:
            return dict(family=family, count=1, n=_log(rng, 100, 4000), conv=rng.choice(CHAR),
                        rk=rng.choice(["rk3", "ls3"]), steps=rng.choice([20, 50, 51]))
        return dict(family=family, count=_log(rng, 8, 300), n=_log(rng, 400, 3000), conv=rng.choice(CHAR),
                    rk=rng.choice(["rk3", "ls3"]), steps=0)
    return dict(family=family, n=_log(rng, 64, 480), conv=rng.choice(["weno_z", "central_skew"]),
                viscous=rng.random() < 0.5, steps=10, every=rng.choice([4, 5, 10]))


# ---------------------------------------------------------------------------
# problems and inputs
# ---------------------------------------------------------------------------
def _axes(n, delta):
    """Coordinates i*delta of every direction, shaped to broadcast (z, y, x)."""
    nd = len(n)
    out = []
    for d in range(nd):
        shape = [1] * nd
        shape[nd - 1 - d] = n[d]
        out.append((torch.arange(n[d], dtype=F64, device=DEV) * delta[d]).reshape(shape))
    return out


def _conserved(rho, u, p, gama):
    rho = rho + torch.zeros_like(sum(u) + p)
    ke = sum(v * v for v in u)
    return torch.stack([rho] + [rho * v for v in u] + [p / (gama - 1.0) + 0.5 * rho * ke]).contiguous()


def _tgv(case, rng):
    n = [case["nx"], case["ny"], case["nz"]]
    delta = [2.0 * math.pi / k for k in n]
    gama, minf = 1.4, 0.1
    problem = dict(ndim=3, n=n, delta=delta, conv=case["conv"], averaging=case["avg"], viscous="const",
                   rk=case["rk"], bc=[["periodic", "periodic"]] * 3, gama=gama, Minf=minf, Re=1600.0, Pr=0.71,
                   dt=3.385e-3 * 64.0 / max(n), eps=1e-16, teno_ct=1e-6)
    X, Y, Z = _axes(n, delta)
    # the vortex, shifted, under a few solenoidal modes u_a(x_b), a != b
    sx, sy, sz = (rng.uniform(0, 2 * math.pi) for _ in range(3))
    x, y, z = X + sx, Y + sy, Z + sz
    u = [torch.sin(x) * torch.cos(y) * torch.cos(z), -torch.cos(x) * torch.sin(y) * torch.cos(z),
         torch.zeros_like(x * y * z)]
    for _ in range(6):
        a, b = rng.sample(range(3), 2)
        k, amp, ph = rng.randint(1, 4), 0.1 * rng.random(), rng.uniform(0, 2 * math.pi)
        u[a] = u[a] + amp * torch.sin(k * (X, Y, Z)[b] + ph)
    p = 1.0 / (gama * minf * minf) + (torch.cos(2 * x) + torch.cos(2 * y)) * (2.0 + torch.cos(2 * z)) / 16.0
    return problem, _conserved(gama * minf * minf * p, u, p, gama)


def _wave(case, rng):
    n = [case["nx"], case["ny"]]
    delta = [2.0 / k for k in n]
    gama = 1.4
    problem = dict(ndim=2, n=n, delta=delta, conv=case["conv"], averaging=case["avg"], viscous="none",
                   rk=case["rk"], bc=[["periodic", "periodic"]] * 2, gama=gama, dt=0.1 * min(delta), eps=1e-16,
                   teno_ct=1e-6)
    X, Y = _axes(n, delta)
    rho = 1.0 + 0.2 * torch.sin(math.pi * (X + Y) + rng.uniform(0, 6)) + \
        0.05 * torch.sin(2 * math.pi * (X - 2 * Y) + rng.uniform(0, 6))
    one = torch.ones_like(rho)
    vel = [one * 1.0 + 0.05 * torch.sin(math.pi * Y + rng.uniform(0, 6)), -0.5 * one]
    return problem, _conserved(rho, vel, one, gama)


def _plate(case, seed):
    nd = 3 if case["nz"] else 2
    n = (case["nx"], case["ny"], case["nz"])[:nd]
    sinh = case["sensor"]  # the Katzer grid; the other plates take the tanh map
    problem, q0 = flat_plate(n=n, lengths=(400.0, 115.0, 35.0), conv=case["conv"], noise=0.0, sensor=case["sensor"],
                             wall=case["wall"], Twall=1.67619431 if case["wall"] == "isothermal_wall" else None,
                             stretch="sinh" if sinh else "tanh", ndim=nd)
    prof = torch.from_numpy(q0[(slice(None),) + (0,) * (nd - 2) + (slice(None), 0)].copy()).to(DEV)
    del q0
    prof = prof.reshape((nd + 2,) + (1,) * (nd - 2) + (n[1], 1)).expand((nd + 2,) + tuple(reversed(n)))
    g = torch.Generator(device=DEV).manual_seed(seed)
    vel = [prof[1 + m] / prof[0] + 1e-3 * torch.randn(prof.shape[1:], dtype=F64, device=DEV, generator=g)
           for m in range(nd)]
    p = 0.4 * (prof[-1] - 0.5 * sum(prof[1 + m] ** 2 for m in range(nd)) / prof[0])
    q = _conserved(prof[0], vel, p, 1.4)
    q[1:nd + 1, ..., 0, :] = 0.0  # the wall is at rest
    return problem, q


def _curv(case, rng):
    make = euler_wave_curvilinear if case["ndim"] == 2 else euler_wave_curvilinear_3d
    problem, q0 = make(case["n"], conv=case["conv"], averaging=case["avg"], dt=0.2 / case["n"])
    q = torch.from_numpy(q0).to(DEV)
    k, ph = rng.randint(1, 3), rng.uniform(0, 6)
    x = _axes(problem["n"], problem["delta"])
    f = 1.0 + 0.1 * torch.sin(math.pi * k * (x[0] - x[1]) + ph)
    return problem, (q * f).contiguous()  # scales density, momentum and energy alike


def _tubes(case, seed):
    """Parameters of the tubes: their sizes belong to the case, the states to the seed."""
    count, top = case["count"], case["n"]
    t_end = 0.2 if count == 1 else 0.04
    par = ensemble_parameters(count, seed=seed % (1 << 31), nmin=top, nmax=top, t_end=t_end)
    if count > 1:
        speed = par["cfl"] * par["dx"] / par["dt"]
        n = np.random.RandomState(3).randint(top // 20, top + 1, size=count)
        dx = 1.0 / (n - 1)
        dt = par["cfl"] * dx / speed
        par.update(n=n.astype(np.int32), dx=dx, dt=dt, nsteps=np.ceil(t_end / dt).astype(np.int64))
    return par


def _kh(case, seed):
    amps = np.random.RandomState(seed % (1 << 31)).normal(0.0, 1e-2, 16)
    problem, q0 = kelvin_helmholtz(case["n"], amps, conv=case["conv"])
    if case["viscous"]:
        problem.update(viscous="const", Re=1000.0, Pr=0.72, Minf=0.5)
    return problem, torch.from_numpy(q0).to(DEV)


def _inputs(case, seed):
    rng = random.Random(seed)
    family = case["family"]
    if family == "tgv":
        return _tgv(case, rng)
    if family == "wave":
        return _wave(case, rng)
    if family == "plate":
        return _plate(case, seed)
    if family == "curv":
        return _curv(case, rng)
    if family == "adjoint":
        return _kh(case, seed)
    par = _tubes(case, seed)
    problem, q = instance_problem(par, 0, case["conv"], case["rk"])
    return problem, torch.from_numpy(q).to(DEV)


def prepare(case, seed):
    if case["family"] == "tubes" and case["count"] > 1:
        e = Ensemble(_tubes(case, seed), case["conv"], case["rk"])
        e.save()
        return dict(case=case, ensemble=e)
    problem, q0 = _inputs(case, seed)
    block = Block(problem)
    q = torch.empty_like(q0)
    torch.cuda.synchronize()  # the block works on a stream of its own
    return dict(case=case, problem=problem, block=block, q0=q0, q=q,
                src=[v.data_ptr() for v in q0], dst=[v.data_ptr() for v in q])


def run(state):
    case = state["case"]
    if case["family"] == "tubes" and case["count"] > 1:
        e = state["ensemble"]
        e.restore()
        e.run("persistent")
        return np.concatenate([e.get_state(i).ravel() for i in range(e.ninst)])
    block = state["block"]
    if case["family"] == "adjoint":
        q0 = state["q0"].detach().requires_grad_(True)
        q = adjoint.integrate(q0, block, case["steps"], case["every"])
        adjoint.kinetic_energy(q, state["problem"]).backward()
        return {"q": q.detach(), "grad": q0.grad}
    block.set_state_dev(state["src"])
    block.run(case["steps"])
    block.get_state_dev(state["dst"])
    return state["q"]


def work(case):
    """Bytes: the state read and written once per pass while it and the RK
    register stay in the 256 MB last-level cache, once per RK stage, with the
    register, where they cannot.  Operations: the schemes' formulas (an
    interface flux, the viscous terms, the update); the adjoint does about
    three times the forward's work."""
    family = case["family"]
    if family == "tubes":
        par = _tubes(case, 1)
        nd, conv, visc = 1, case["conv"], False
        steps = np.full(1, case["steps"]) if case["count"] == 1 else par["nsteps"]
        cells = float(np.sum(par["n"]))
        updates = 3.0 * float(np.sum(par["n"].astype(np.float64) * steps))
    else:
        if family in ("tgv", "wave", "plate"):
            n = [case["nx"], case["ny"]] + ([case["nz"]] if case.get("nz") else [])
        elif family == "curv":
            n = [case["n"]] * case["ndim"]
        else:
            n = [case["n"]] * 2
        nd, conv = len(n), case["conv"]
        visc = family in ("tgv", "plate") or bool(case.get("viscous"))
        cells = float(np.prod([float(k) for k in n]))
        updates = 3.0 * cells * case["steps"]
    nv = nd + 2
    if conv.startswith("central"):
        flops = nd * (80.0, 110.0, 140.0)[nd - 1]
    else:
        recon = {"weno_z": 76.0, "weno_js": 70.0, "teno5": 88.0, "teno6": 100.0}[conv]
        flops = nd * ((300.0, 620.0, 850.0)[nd - 1] + 2 * nv * (recon + 1.0))
    flops += 12.0 * nv + ((40.0, 200.0, 530.0)[nd - 1] if visc else 0.0)
    fields = 2.0 * nv + (nd * nd + 1 if family == "curv" else 0)
    if 8.0 * fields * cells > 256e6:
        nbytes = 8.0 * (fields + 2.0 * nv) * updates
    else:
        nbytes = 16.0 * nv * cells
    if family == "adjoint":
        nbytes, flops = 2.0 * nbytes, 3.0 * flops
    return dict(bytes=nbytes, flops=flops * updates)


# ---------------------------------------------------------------------------
# the schemes in plain torch, on arrays padded by H points in every direction;
# direction d is tensor axis -1 - d
# ---------------------------------------------------------------------------
H = 4
RK3 = ([2.0 / 3.0, 5.0 / 12.0, 3.0 / 5.0], [1.0 / 4.0, 3.0 / 20.0, 3.0 / 5.0])
LS3 = ([0.0, -5.0 / 9.0, -153.0 / 128.0], [1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0])


def _sh(f, k, axis):
    return f if not torch.is_tensor(f) else torch.roll(f, -k, axis)


def _weno(v, js):
    fm2, fm1, f0, f1, f2 = v
    b = [13.0 / 12.0 * (f0 - 2 * f1 + f2) ** 2 + 0.25 * (3 * f0 - 4 * f1 + f2) ** 2,
         13.0 / 12.0 * (fm1 - 2 * f0 + f1) ** 2 + 0.25 * (fm1 - f1) ** 2,
         13.0 / 12.0 * (fm2 - 2 * fm1 + f0) ** 2 + 0.25 * (fm2 - 4 * fm1 + 3 * f0) ** 2]
    d = (0.3, 0.6, 0.1)
    if js:
        w = [d[r] / (1e-6 + b[r]) ** 2 for r in range(3)]
    else:
        tau = torch.abs(b[0] - b[2])
        w = [d[r] * (1.0 + (tau / (1e-14 + b[r])) ** 2) for r in range(3)]
    c = [(2 * f0 + 5 * f1 - f2) / 6, (-fm1 + 5 * f0 + 2 * f1) / 6, (2 * fm2 - 7 * fm1 + 11 * f0) / 6]
    return sum(w[r] * c[r] for r in range(3)) / sum(w)


def _teno(v, eps, ct, six, right):
    fm2, fm1, f0, f1, f2, f3 = v
    b = [0.25 * (fm1 - f1) ** 2 + 13.0 / 12.0 * (fm1 - 2 * f0 + f1) ** 2,
         0.25 * (3 * f0 - 4 * f1 + f2) ** 2 + 13.0 / 12.0 * (f0 - 2 * f1 + f2) ** 2,
         0.25 * (fm2 - 4 * fm1 + 3 * f0) ** 2 + 13.0 / 12.0 * (fm2 - 2 * fm1 + f0) ** 2]
    c = [(-fm1 + 5 * f0 + 2 * f1) / 6, (2 * f0 + 5 * f1 - f2) / 6, (2 * fm2 - 7 * fm1 + 11 * f0) / 6]
    if six:
        t = -f0 + 3 * f1 - 3 * f2 + f3
        # the right-hand indicator's last term is not squared, as published in the reference (teno.py:166-167)
        b.append((-11 * f0 + 18 * f1 - 9 * f2 + 2 * f3) ** 2 / 36.0 +
                 13.0 / 12.0 * (2 * f0 - 5 * f1 + 4 * f2 - f3) ** 2 + 781.0 / 720.0 * (t if right else t * t))
        c.append((3 * f0 + 13 * f1 - 5 * f2 + f3) / 12)
        tau = torch.abs(b[3] - (b[0] + b[2] - 4 * b[1]) / 6)
        d = (231.0 / 500.0, 3.0 / 10.0, 27.0 / 500.0, 23.0 / 125.0)
    else:
        tau = torch.abs(b[0] - b[2])
        d = (11.0 / 20.0, 4.0 / 10.0, 1.0 / 20.0)
    a = [(1.0 + tau / (eps + x)) ** 6 for x in b]
    s = sum(a)
    w = [dr * (x / s >= ct).to(F64) for dr, x in zip(d, a)]
    return sum(x * y for x, y in zip(w, c)) / sum(w)


def _pair(p, conv, fp, fm, ct):
    if conv in ("weno_z", "weno_js"):
        return _weno(fp[:5], conv == "weno_js") + _weno(fm[:0:-1], conv == "weno_js")
    six, eps = conv == "teno6", p.get("eps", 1e-16)
    return _teno(fp, eps, ct, six, True) + _teno(fm[::-1], eps, ct, six, False)


def _eigen(nd, k, u, rho, a, gama):
    """Rows of L and columns of R of the Euler Jacobian about the unit normal k."""
    gm1 = gama - 1.0
    phi = 0.5 * gm1 * sum(v * v for v in u)
    if nd == 1:
        v, h = u[0], a * a / gm1 + 0.5 * u[0] ** 2
        den = 2 * h - v * v
        L = [[v * (2 * h + a * v - v * v) / (2 * a * den), (-h - a * v + 0.5 * v * v) / (a * den), 1 / den],
             [2 * (h - v * v) / den, 2 * v / den, -2 / den],
             [v * (-2 * h + a * v + v * v) / (2 * a * den), (h - a * v - 0.5 * v * v) / (a * den), 1 / den]]
        R = [[1.0, v - a, h - v * a], [1.0, v, 0.5 * v * v], [1.0, v + a, h + v * a]]
        return L, R
    th = sum(x * y for x, y in zip(k, u))
    al, be = rho / (math.sqrt(2.0) * a), 1.0 / (math.sqrt(2.0) * rho * a)
    ent = [1.0 - phi / a ** 2] + [gm1 * v / a ** 2 for v in u] + [-gm1 / a ** 2]
    entr = [1.0] + list(u) + [phi / gm1]
    L, R = [], []
    if nd == 2:
        c = k[1] * u[0] - k[0] * u[1]
        L = [ent, [-c / rho, k[1] / rho, -k[0] / rho, 0.0]]
        R = [entr, [0.0, k[1] * rho, -k[0] * rho, rho * c]]
    else:
        cr = [k[1] * u[2] - k[2] * u[1], k[2] * u[0] - k[0] * u[2], k[0] * u[1] - k[1] * u[0]]
        for f in range(3):
            e = [0.0, 0.0, 0.0]
            e[(f + 1) % 3], e[(f + 2) % 3] = k[(f + 2) % 3], -1.0 * k[(f + 1) % 3]
            L.append([k[f] * ent[0] + cr[f] / rho] + [k[f] * ent[1 + c] + e[c] / rho for c in range(3)] +
                     [k[f] * ent[4]])
            R.append([k[f] * entr[0]] + [k[f] * entr[1 + c] + rho * e[c] for c in range(3)] +
                     [k[f] * entr[4] - rho * cr[f]])
    for s in (1.0, -1.0):
        L.append([be * (phi - s * a * th)] + [be * (s * k[c] * a - gm1 * u[c]) for c in range(nd)] + [be * gm1])
        R.append([al] + [al * (u[c] + s * k[c] * a) for c in range(nd)] + [al * ((phi + a * a) / gm1 + s * a * th)])
    return L, R


def _char_flux(p, q, d, ct, metric=None):
    """LLF characteristic flux at i + 1/2 along d, stored at i."""
    nd, gama, conv = p["ndim"], p["gama"], p["conv"]
    nv, ax, gm1 = nd + 2, -1 - d, gama - 1.0
    u = [q[1 + m] / q[0] for m in range(nd)]
    pr = gm1 * (q[-1] - 0.5 * q[0] * sum(v * v for v in u))
    a = torch.sqrt(gama * pr / q[0])
    if metric is None:
        k, km, dj = [1.0 if m == d else 0.0 for m in range(nd)], 1.0, 1.0
        kt = k
    else:
        k, dj = metric["D"][d], metric["detJ"]
        km = torch.sqrt(sum(x * x for x in k))
        kt = [0.5 * (x + _sh(x, 1, ax)) for x in k]
        norm = torch.sqrt(sum(x * x for x in kt))
        kt = [x / norm for x in kt]
    U = u[d] if metric is None else sum(x * y for x, y in zip(k, u))
    F = [dj * q[0] * U] + [dj * (q[1 + m] * U + pr * k[m]) for m in range(nd)] + [dj * (pr + q[-1]) * U]
    if p["averaging"] == "roe":
        s = torch.sqrt(q[0])
        s1 = _sh(s, 1, ax)
        mean = lambda f: (s * f + s1 * _sh(f, 1, ax)) / (s + s1)  # noqa: E731
        ua, ha = [mean(v) for v in u], mean((q[-1] + pr) / q[0])
        ra, aa = s * s1, torch.sqrt(gm1 * (ha - 0.5 * sum(v * v for v in ua)))
    else:
        mean = lambda f: 0.5 * (f + _sh(f, 1, ax))  # noqa: E731
        ua, ra, aa = [mean(v) for v in u], mean(q[0]), mean(a)
    L, R = _eigen(nd, kt, ua, ra, aa, gama)
    speeds = [U - a, U, U + a] if nd == 1 else [U] * nd + [U + a * km, U - a * km]
    out = [0.0] * nv
    for f in range(nv):
        w = torch.abs(speeds[f])
        lam = _sh(w, -2, ax)
        for s in range(-1, 4):
            nxt = _sh(w, s, ax)
            lam = torch.where(nxt > lam, nxt, lam)
        fp, fm = [], []
        for s in range(-2, 4):
            cf = sum(L[f][m] * _sh(F[m], s, ax) for m in range(nv))
            cs = sum(L[f][m] * _sh(q[m], s, ax) for m in range(nv))
            fp.append(0.5 * (cf + lam * cs))
            fm.append(0.5 * (cf - lam * cs))
        rec = _pair(p, conv, fp, fm, ct)
        out = [o + R[f][m] * rec for m, o in enumerate(out)]
    return out


def _closure_rows(order, scheme):
    """One-sided rows of the central first / second derivative at a closed face."""
    if order == 2:
        return [[35 / 12, -104 / 12, 114 / 12, -56 / 12, 11 / 12], [11 / 12, -20 / 12, 6 / 12, 4 / 12, -1 / 12]]
    assert scheme == "reduced_access"
    return [[-25 / 12, 48 / 12, -36 / 12, 16 / 12, -3 / 12], [-3 / 12, -10 / 12, 18 / 12, -6 / 12, 1 / 12]]


def _closed(p, d, side):
    return p["bc"][d][side] not in ("periodic", "zero_gradient", "symmetry")


def _deriv(p, f, d, order):
    """Central derivative along d in the computational coordinate, with the faces' closures."""
    ax = -1 - d
    if order == 1:
        r = (_sh(f, -2, ax) - _sh(f, 2, ax)) / 12 + 2.0 / 3.0 * (_sh(f, 1, ax) - _sh(f, -1, ax))
    else:
        r = -(_sh(f, -2, ax) + _sh(f, 2, ax)) / 12 + 4.0 / 3.0 * (_sh(f, 1, ax) + _sh(f, -1, ax)) - 2.5 * f
    n = p["n"][d]
    for side in (0, 1):
        if not _closed(p, d, side):
            continue
        for c, row in enumerate(_closure_rows(order, p["bscheme"][d][side])):
            at = [H + j if side == 0 else H + n - 1 - j for j in range(len(row))]
            v = sum(w * f.select(ax, i) for w, i in zip(row, at))
            r.select(ax, at[c]).copy_(-v if order == 1 and side else v)
    return r / p["delta"][d] ** order


def _stretch(p, d):
    """D_dd and SD_ddd of a stretched direction over the padded line, mirrored in the halos; None otherwise."""
    if not p.get("stretch", [0, 0, 0])[d]:
        return None
    line = dict(p, n=[p["n"][d]], delta=[p["delta"][d]], bc=[p["bc"][d]], bscheme=[p["bscheme"][d]])
    x = torch.nn.functional.pad(torch.from_numpy(np.asarray(p["coords"][d])).to(DEV), (H, H))
    G = 1.0 / _deriv(line, x, 0, 1)
    S = _deriv(line, G, 0, 1)
    for f in (G, S):
        for h in range(1, H + 1):
            f[H - h], f[-1 - H + h] = f[H + h], f[-1 - H - h]
    shape = [1] * p["ndim"]
    shape[-1 - d] = -1
    return G.reshape(shape), S.reshape(shape)


def _viscous(p, q, prims, met):
    nd = p["ndim"]
    u, T = prims["u"], prims["T"]
    mu = prims.get("mu")
    inv_re, cq = 1.0 / p["Re"], 1.0 / ((p["gama"] - 1.0) * p["Minf"] ** 2 * p["Pr"] * p["Re"])
    G = [m[0] if m else 1.0 for m in met]

    def first(f, j):
        return G[j] * _deriv(p, f, j, 1)

    def second(f, j):
        v = _deriv(p, f, j, 2)
        return G[j] * G[j] * v + G[j] * met[j][1] * _deriv(p, f, j, 1) if met[j] else v

    du = [[first(u[m], j) for j in range(nd)] for m in range(nd)]
    dd = {}
    for m in range(nd):
        for a in range(nd):
            dd[m, a, a] = second(u[m], a)
            for b in range(a + 1, nd):
                if m in (a, b):
                    dd[m, a, b] = dd[m, b, a] = G[a] * G[b] * _deriv(p, _deriv(p, u[m], a, 1), b, 1)
    div = sum(du[m][m] for m in range(nd))
    energy = 0.0
    for j in range(nd):
        t = second(T, j)
        energy = energy + cq * (t if mu is None else mu * t + first(mu, j) * first(T, j))
    r = [torch.zeros_like(T)]
    for m in range(nd):
        total = 0.0
        for j in range(nd):
            tt = dd[m, j, j] + dd[j, m, j]
            sr = du[m][j] + du[j][m]
            if j == m:
                tt = tt - 2.0 / 3.0 * sum(dd[k, m, k] for k in range(nd))
                sr = sr - 2.0 / 3.0 * div
            dtau = inv_re * tt if mu is None else inv_re * (mu * tt + first(mu, j) * sr)
            tau = inv_re * sr if mu is None else inv_re * mu * sr
            total = total + dtau
            energy = energy + du[m][j] * tau + u[m] * dtau
        r.append(total)
    return r + [energy]


def _central(p, q, prims):
    nd, nv = p["ndim"], p["ndim"] + 2
    u, pr = prims["u"], prims["p"]
    r = [torch.zeros_like(pr) for _ in range(nv)]
    for j in range(nd):
        D = lambda f: _deriv(p, f, j, 1)  # noqa: E731
        if p["conv"] == "central_skew":
            duj = D(u[j])
            for m in range(nv):
                r[m] = r[m] - 0.5 * (D(q[m] * u[j]) + u[j] * D(q[m]) + q[m] * duj)
            r[1 + j] = r[1 + j] - D(pr)
            r[-1] = r[-1] - D(pr * u[j])
        else:
            r[0] = r[0] - D(q[1 + j])
            for m in range(nd):
                r[1 + m] = r[1 + m] - D(q[1 + m] * u[j] + (pr if m == j else 0.0))
            r[-1] = r[-1] - D((pr + q[-1]) * u[j])
    return r


def _sensor_ct(p, u, met):
    """Adaptive TENO cut-off from the modified Ducros sensor at every point."""
    nd = p["ndim"]
    du = [[(met[d][0] if met[d] else 1.0) * _deriv(p, u[m], d, 1) for d in range(nd)] for m in range(nd)]
    div = sum(du[m][m] for m in range(nd))
    w = [du[1][0] - du[0][1]]
    if nd == 3:
        w += [du[2][1] - du[1][2], du[0][2] - du[2][0]]
    th = 0.5 * (1.0 - torch.tanh(2.5 * (1.0 + 100.0 * div))) * div ** 2 / \
        (div ** 2 + sum(x * x for x in w) + p["sensor_eps"])
    beta = p["teno_a1"] - p["teno_a2"] * (1.0 - (1.0 - th) ** 4 * (1.0 + 4.0 * th))
    return 10.0 ** -torch.floor(beta)


def _rhs(p, q, met, metric=None):
    """Residual on the padded arrays (right on the interior)."""
    nd, gm1 = p["ndim"], p["gama"] - 1.0
    visc = p.get("viscous", "none")
    u = [q[1 + m] / q[0] for m in range(nd)]
    prims = {"u": u, "p": gm1 * (q[-1] - 0.5 * q[0] * sum(v * v for v in u))}
    if p["conv"].startswith("central"):
        r = _central(p, q, prims)
    else:
        ct = _sensor_ct(p, u, met) if p.get("sensor") else p.get("teno_ct", 1e-6)
        r = [0.0] * (nd + 2)
        for d in range(nd):
            F = _char_flux(p, q, d, ct, metric)
            G = met[d][0] if met[d] else 1.0
            r = [x - G * (f - _sh(f, -1, -1 - d)) / p["delta"][d] for x, f in zip(r, F)]
        if metric is not None:
            r = [x / metric["detJ"] for x in r]
    if visc != "none":
        prims["T"] = prims["p"] * p["gama"] * p["Minf"] ** 2 / q[0]
        if visc == "sutherland":
            s = p["SuthT"] / p["RefT"]
            prims["mu"] = prims["T"] ** 1.5 * (1.0 + s) / (prims["T"] + s)
        r = [x + y for x, y in zip(r, _viscous(p, q, prims, met))]
    return torch.stack(r)


def _face(p, q, d, side):
    """One non-periodic face, in place."""
    nd, ax, n, gama = p["ndim"], -1 - d, p["n"][d], p["gama"]
    gm1, M2, bc = gama - 1.0, p["Minf"] ** 2, p["bc"][d][side]
    at = lambda i: q.select(ax, H + i if side == 0 else H + n - 1 - i)  # noqa: E731, i inward
    temp = lambda s: (s[-1] - 0.5 * sum(s[1:-1] ** 2) / s[0]) * gama * gm1 * M2 / s[0]  # noqa: E731
    if bc == "extrap0":
        for h in range(H + 1):
            at(-h).copy_(at(1))
    elif bc == "dirichlet":
        plane = torch.from_numpy(np.asarray(p["planes"][d, side])).to(DEV)  # (nv, e2, e1)
        shape = list(at(0).shape)
        idx = [torch.arange(-H, k - H, device=DEV).clamp(0, m - 1) for k, m in
               zip(shape[1:], plane.shape[-len(shape) + 1:])]
        plane = plane.reshape((nd + 2,) + tuple(plane.shape[-len(shape) + 1:]))
        for a, i in enumerate(idx):
            plane = plane.index_select(1 + a, i)
        for h in range(H + 1):
            at(-h).copy_(plane)
    elif bc == "inlet_pextrap":
        s = at(0).clone()
        ke = sum((s[1 + m] / s[0]) ** 2 for m in range(nd))
        a = torch.sqrt(gama * gm1 * (s[-1] - 0.5 * s[0] * ke) / s[0])
        sup = torch.abs(s[1 + d] / s[0]) >= a
        at(0).copy_(torch.where(sup, at(-1), s))
        for h in range(1, H + 1):
            at(-h)[-1].copy_(torch.where(sup, at(-h)[-1], s[-1]))
    else:
        w = at(0)
        w[1:-1] = 0.0
        if bc == "adiabatic_wall":
            T = [temp(at(i)) for i in (1, 2, 3)]
            w[-1] = w[0] * (6.0 / 11.0) * (3.0 * T[0] + T[2] / 3.0 - 1.5 * T[1]) / (gama * M2) / gm1
            for h in range(1, H + 1):
                at(-h).copy_(at(h))
                at(-h)[1:-1] *= -1.0
        else:
            tw = p["Twall"]
            w[-1] = w[0] * tw / (gama * gm1 * M2)
            pw, Ta = gm1 * w[-1], temp(at(1))
            for h in range(1, H + 1):
                s = at(h)
                vel = [s[1 + m] / s[0] for m in range(nd)]
                r = pw * gama * M2 / ((h + 1) * tw - h * Ta)
                at(-h).copy_(torch.stack([r] + [-r * v for v in vel] +
                                         [pw / gm1 + 0.5 * r * sum(v * v for v in vel)]))


def _fill(p, q):
    """Boundary conditions on the padded state, direction by direction."""
    for d in range(p["ndim"]):
        ax, n = -1 - d, p["n"][d]
        if p["bc"][d][0] == "periodic":
            idx = (torch.arange(-H, n + H, device=q.device) % n) + H
            q = q.index_select(q.dim() + ax, idx)
        else:
            q = q.clone()
            for side in (0, 1):
                _face(p, q, d, side)
    return q


def _inside(p, q):
    for d in range(p["ndim"]):
        q = q.narrow(-1 - d, H, p["n"][d])
    return q


def _step(p, q, fill, rhs, dt):
    A, B = RK3 if p["rk"] == "rk3" else LS3
    old = q if p["rk"] == "rk3" else torch.zeros_like(q)
    for a, b in zip(A, B):
        r = dt * rhs(q)
        if p["rk"] == "rk3":
            q, old = fill(old + a * r, q), old + b * r
        else:
            old = a * old + r
            q = fill(q + b * old, q)
    return q


def _advance(p, q0, steps):
    """`steps` iterations of the problem from the interior state q0; the interior afterwards."""
    nd = p["ndim"]
    pad = (H, H) * nd
    q = torch.nn.functional.pad(q0, pad)
    outside = None
    if any(side == "inlet_pextrap" for face in p["bc"] for side in face):
        plane = torch.from_numpy(np.asarray(p["planes"][0, 0])).to(DEV)
        plane = plane.reshape((nd + 2,) + tuple(plane.shape[-nd + 1:]) + (1,))
        v = q[(slice(None),) + (slice(H, -H),) * (nd - 1) + (slice(0, H),)]
        v.copy_(plane.expand_as(v))
        outside = True
    met = [_stretch(p, d) for d in range(nd)]
    metric = _metric(p) if p.get("curvilinear") else None

    def fill(new, prev):
        if outside is None:
            return _fill(p, new)
        keep = prev.clone()  # the inlet's halos persist
        _inside(p, keep).copy_(_inside(p, new))
        return _fill(p, keep)

    def rhs(state):
        return _rhs(p, state, met, metric)

    q = _fill(p, q)
    for _ in range(steps):
        if torch.is_grad_enabled():
            q = torch.utils.checkpoint.checkpoint(lambda s: _step(p, s, fill, rhs, p["dt"]), q, use_reentrant=False)
        else:
            q = _step(p, q, fill, rhs, p["dt"])
    return _inside(p, q)


def _metric(p):
    """D_ab = d xi_a / d x_b and detJ from the grid coordinates, with periodic halos."""
    nd, g = p["ndim"], p["grid_halo"]
    X = torch.from_numpy(np.asarray(p["grid_coords"])).to(DEV)
    J = torch.zeros((nd, nd) + tuple(n for n in reversed(p["n"])), dtype=F64, device=DEV)
    for b in range(nd):
        D = (_sh(X, -2, -1 - b) - _sh(X, 2, -1 - b)) / 12 + 2.0 / 3.0 * (_sh(X, 1, -1 - b) - _sh(X, -1, -1 - b))
        for d in range(nd):
            D = D.narrow(-1 - d, g, p["n"][d])
        J[:, b] = D / p["delta"][b]
    m = torch.movedim(J, (0, 1), (-2, -1))
    det = torch.linalg.det(m)
    inv = torch.movedim(torch.linalg.inv(m), (-2, -1), (0, 1))
    flat = _fill(p, torch.nn.functional.pad(torch.cat([inv.flatten(0, 1), det[None]]), (H, H) * nd))
    return {"D": [[flat[a * nd + b] for b in range(nd)] for a in range(nd)], "detJ": flat[-1]}


def _exact_tubes(case, seed):
    """Every tube as a row of one padded array; zeroth-order ends are an index clamp."""
    par = _tubes(case, seed)
    count = case["count"]
    top = int(par["n"].max())
    n = torch.from_numpy(par["n"].astype(np.int64)).to(DEV)[:, None]
    q = torch.ones((3, count, top), dtype=F64, device=DEV)
    for i in range(count):
        p, s = instance_problem(par, i, case["conv"], case["rk"])
        q[:, i, :p["n"][0]] = torch.from_numpy(s)
    steps = torch.full_like(n, case["steps"]) if count == 1 else torch.from_numpy(par["nsteps"]).to(DEV)[:, None]
    dt, dx = (torch.from_numpy(np.asarray(par[k])).to(DEV)[:, None] for k in ("dt", "dx"))
    p = dict(p, delta=[dx], n=[top])
    idx = torch.minimum(torch.arange(-H, top + H, device=DEV)[None].clamp(min=1), n - 2) + H

    def fill(new, prev):
        return torch.gather(new, 2, idx.expand_as(new))

    q = fill(torch.nn.functional.pad(q, (H, H)), None)
    for s in range(int(steps.max())):
        q = torch.where(s < steps, _step(p, q, fill, lambda x: _rhs(p, x, [None]), dt), q)
    q = q[..., H:-H]
    if count == 1:
        return q[:, 0].contiguous()
    return np.concatenate([q[:, i, :int(par["n"][i])].cpu().numpy().ravel() for i in range(count)])


def exact(case, seed):
    if case["family"] == "tubes":
        with torch.no_grad():
            return _exact_tubes(case, seed)
    problem, q0 = _inputs(case, seed)
    if case["family"] == "adjoint":
        q0.requires_grad_(True)
        q = _advance(problem, q0, case["steps"])
        adjoint_dv = problem["delta"][0] * problem["delta"][1]
        (0.5 * ((q[1] ** 2 + q[2] ** 2) / q[0]).sum() * adjoint_dv).backward()
        return {"q": q.detach(), "grad": q0.grad}
    with torch.no_grad():
        return _advance(problem, q0, case["steps"])
