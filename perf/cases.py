"""Timed cases: what a program does with this engine, through its public entry points.

A case is one kind of call at one size (the kinds are described at `listed`).
Inputs are seeded synthetic systems of the benchmark's distributions: Plummer
spheres, two colliding spheres, ensembles of clusters and of planetary systems,
a disc around a star.  FP64-state runs return the state as it is held; where the
pair arithmetic or the state is single precision and the caller asks for forces,
potentials or an FP32 state, the caller keeps them in single precision too.
"""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

from __graft_entry__ import load_package

nb = load_package()

FLOPS_PER_PAIR = 20.0


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # A small system integrated step by step (a binary's cluster, a test
        # run): launches and latency count, the arithmetic hardly does.
        {"name": "steps_split_1000", "kind": "steps", "mode": "split", "n": 1000, "steps": 64, "h": 0.01},
        # The 4096-body Plummer sphere of the reference's own examples.
        {"name": "steps_split_4096", "kind": "steps", "mode": "split", "n": 4096, "steps": 32, "h": 0.01},
        # A single-precision run (the reference's floattype = Float32 on GPU).
        {"name": "steps_fp32_65536", "kind": "steps", "mode": "fp32", "n": 65536, "steps": 4, "h": 0.005},
        # Two spheres of 2^19 bodies on a head-on course: the largest run.
        {"name": "collision_1048576", "kind": "collision", "mode": "split", "n": 1048576, "steps": 1, "h": 0.002},
        # All-FP64 forces, asked for to check another run or to publish.
        {"name": "force_fp64_10007", "kind": "force", "mode": "fp64", "n": 10007, "h": 0.01},
        # An analyser's potential of every particle, at a ragged size.
        {"name": "potential_split_30011", "kind": "potential", "mode": "split", "n": 30011, "h": 0.01},
        # A rotation curve or a field map: the force at points that are not
        # particles, in a large system.
        {"name": "probes_1009_in_200003", "kind": "probes", "mode": "split", "n": 200003, "npts": 1009, "h": 0.01},
        # A whole Simulation with adaptive block steps, made, run and read out
        # as the galaxy-collision example does (60000 bodies, FP32).
        {"name": "adaptive_run_60000", "kind": "adaptive", "mode": "fp32", "n": 60000, "t_end": 1.0, "h": 0.02},
        # 512 clusters of 256 to 16384 bodies in one launch.
        {"name": "clusters_512", "kind": "clusters", "mode": "split", "nsys": 512, "nmin": 256, "nmax": 16384,
         "steps": 8},
        # 2048 planetary systems, many steps, their energies tracked.
        {"name": "planets_2048", "kind": "planets", "mode": "split_central", "nsys": 2048, "nplanets": 8,
         "ntest": 64, "steps": 500, "every": 100},
        # Planetesimals around a star: the star's terms in FP64, the rest split.
        {"name": "disc_split_central_16001", "kind": "disc", "mode": "split_central", "n": 16001, "steps": 8,
         "h": 0.001},
        # A serving loop: forces and potentials of a small system that lives in
        # the caller's device arrays, with no allocation.
        {"name": "device_arrays_fp64_2048", "kind": "device", "mode": "fp64", "n": 2048, "h": 0.01},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "collision", "force", "potential", "probes", "adaptive",
                       "clusters", "planets", "disc", "device"])
    if kind == "steps":
        n = _log(rng, 256, 131072)
        return {"kind": kind, "mode": rng.choice(["split", "fp32"]), "n": n, "steps": max(2, min(64, 131072 // n)),
                "h": rng.choice([0.005, 0.01])}
    if kind == "collision":
        return {"kind": kind, "mode": "split", "n": 2 * _log(rng, 65536, 393216), "steps": 1, "h": 0.002}
    if kind == "force":
        return {"kind": kind, "mode": rng.choice(["fp64", "fp64", "split", "fp32"]), "n": _log(rng, 300, 30000),
                "h": 0.01}
    if kind == "potential":
        return {"kind": kind, "mode": rng.choice(["split", "fp32"]), "n": _log(rng, 1000, 120000), "h": 0.01}
    if kind == "probes":
        return {"kind": kind, "mode": rng.choice(["split", "split", "fp64", "fp32"]), "n": _log(rng, 10000, 400000),
                "npts": _log(rng, 1, 4096), "h": 0.01}
    if kind == "adaptive":
        return {"kind": kind, "mode": rng.choice(["fp32", "split"]), "n": 2 * _log(rng, 2000, 30000),
                "t_end": 1.0, "h": 0.02}
    if kind == "clusters":
        return {"kind": kind, "mode": "split", "nsys": _log(rng, 32, 400), "nmin": 256, "nmax": 16384, "steps": 8}
    if kind == "planets":
        return {"kind": kind, "mode": "split_central", "nsys": _log(rng, 100, 2500),
                "nplanets": rng.randrange(2, 11), "ntest": rng.randrange(0, 100), "steps": 500, "every": 100}
    if kind == "disc":
        return {"kind": kind, "mode": "split_central", "n": _log(rng, 1000, 40000), "steps": 8, "h": 0.001}
    return {"kind": kind, "mode": rng.choice(["fp64", "split"]), "n": _log(rng, 300, 20000), "h": 0.01}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
# Steps short enough for the smallest softening and the closest pairs.
DT = {"steps": 1e-4, "collision": 1e-3, "disc": 1e-3, "clusters": 1.25e-4, "planets": 1e-3}


def _system(case, seed):
    """Positions, velocities and masses of a one-system case (host, FP64)."""
    n = case["n"]
    if case["kind"] in ("collision", "adaptive"):
        return nb.ics.collision(n // 2, (seed, seed + 1))
    if case["kind"] == "disc":
        rng = np.random.Generator(np.random.PCG64(seed))
        r = rng.uniform(0.8, 1.2, n)
        phi = rng.uniform(0.0, 2.0 * math.pi, n)
        v = 1.0 / np.sqrt(r)
        pos = np.stack([r * np.cos(phi), r * np.sin(phi), 0.005 * rng.standard_normal(n)], axis=1)
        vel = np.stack([-v * np.sin(phi), v * np.cos(phi), 0.005 * rng.standard_normal(n)], axis=1)
        mass = np.full(n, 1e-3 / n)
        pos[0], vel[0], mass[0] = 0.0, 0.0, 1.0   # the star
        return pos, vel, mass
    return nb.ics.plummer(n, seed)


def _clusters(case, seed):
    """Offsets, positions, velocities, masses and softening lengths of an ensemble
    (the sizes are the case's, log-uniform; the seed gives the particles)."""
    rng = np.random.Generator(np.random.PCG64(1000 + case["nsys"]))
    nsys = case["nsys"]
    ns = np.rint(np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]), nsys))).astype(np.int64)
    rng = np.random.Generator(np.random.PCG64(seed))
    off = np.zeros(nsys + 1, dtype=np.int64)
    off[1:] = np.cumsum(ns)
    a = rng.uniform(0.5, 2.0, nsys)
    pos, vel, _ = nb.ics.plummer(int(off[-1]), seed)   # one unit sphere, dealt out and scaled
    per = np.repeat(a, ns)[:, None]
    return off, pos * per, vel / np.sqrt(per), np.repeat(1.0 / ns, ns), 0.01 * a


def _points(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed + 77))
    return rng.standard_normal((case["npts"], 3))


def _planets(case, seed):
    return nb.ics.planetary_ensemble(case["nsys"], seed, case["nplanets"], case["ntest"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "clusters":
        off, pos, vel, mass, h = _clusters(case, seed)
        e = nb.Ensemble(off, case["mode"])
        e.set_params(1.0, h, DT[kind])
        e.upload(pos, vel, mass)
        e.compute_force()
        e.half_kick(+1)
        e.sync()
        return {"case": case, "ens": e}
    if kind == "planets":
        p = _planets(case, seed)
        e = nb.Ensemble(p["offsets"], case["mode"])
        e.set_params(1.0, 0.0, DT[kind])
        e.upload(p["pos"], p["vel"], p["mass"])
        e.set_central(1)
        e.compute_force()
        e.half_kick(+1)
        e.sync()
        return {"case": case, "ens": e}
    pos, vel, mass = _system(case, seed)
    if kind == "adaptive":
        return {"case": case, "data": nb.StarData(pos, vel, mass)}
    if kind == "device":
        xyz = torch.from_numpy(np.ascontiguousarray(pos.T)).cuda()
        out = torch.empty((4, case["n"]), dtype=torch.float64, device="cuda")
        return {"case": case, "xyz": xyz, "mass": torch.from_numpy(mass).cuda(), "out": out}
    ctx = nb._native.Context(case["n"], nb._native.MODES[case["mode"]])
    ctx.set_params(1.0, [case["h"]] * 6)
    ctx.upload(pos, vel, mass)
    if kind == "disc":
        ctx.set_central(1)
    state = {"case": case, "ctx": ctx}
    if kind == "probes":
        state["pts"] = _points(case, seed)
    if kind in ("steps", "collision", "disc"):
        ctx.compute_force()
        ctx.half_kick(+1, DT[kind])
    ctx.sync()
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _held(case, v):
    """The caller's copy of a result: single precision where the mode's is."""
    return v if case["mode"] == "fp64" else v.astype(np.float32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("steps", "collision", "disc"):
        ctx = state["ctx"]
        ctx.kdk_steps(case["steps"], DT[kind], 0.0, use_graph=True)
        d = ctx.download(pos=True, vel=True, acc=False)
        if case["mode"] == "fp32":   # an FP32 state
            return [d["pos"].astype(np.float32), d["vel"].astype(np.float32)]
        return [d["pos"], d["vel"]]
    if kind == "clusters":
        e = state["ens"]
        e.kdk_steps(case["steps"])
        d = e.download(pos=True, vel=True, acc=False)
        return [d["pos"], d["vel"]]
    if kind == "planets":
        e = state["ens"]
        energy = e.kdk_steps_tracked(case["steps"], case["every"])
        d = e.download(pos=True, vel=True, acc=False)
        return [energy, d["pos"], d["vel"]]
    if kind == "force":
        ctx = state["ctx"]
        ctx.compute_force()
        return [_held(case, ctx.download(pos=False, vel=False, acc=True)["acc"])]
    if kind == "potential":
        ctx = state["ctx"]
        ctx.compute_potential()
        return [_held(case, ctx.download(pos=False, vel=False, acc=False, pot=True)["pot"])]
    if kind == "probes":
        return [_held(case, state["ctx"].force_at_points(state["pts"], case["h"]))]
    if kind == "adaptive":
        sim = nb.Simulation(state["data"], precision=case["mode"], TimeEnd=case["t_end"],
                            TimeBetweenSnapshots=2.0 * case["t_end"], ForceSofteningTable=case["h"],
                            OutputDir=os.path.join(tempfile.gettempdir(), "nbody_cases"),
                            output_func=lambda s: None)
        try:
            nb.run(sim)
            d = nb.get_all_data(sim)
        finally:
            sim.close()
        return [d.Pos.astype(np.float32), d.Vel.astype(np.float32)]
    xyz, out = state["xyz"], state["out"]
    row = out.stride(0) * out.element_size()
    at = out.data_ptr()
    nb._native.compute_force_noalloc(
        nb._native.MODES[case["mode"]], case["n"], xyz[0].data_ptr(), xyz[1].data_ptr(), xyz[2].data_ptr(),
        state["mass"].data_ptr(), at, at + row, at + 2 * row, at + 3 * row, h_const=case["h"],
        stream=torch.cuda.current_stream().cuda_stream)
    return [out if case["mode"] == "fp64" else out.float()]


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "clusters":
        lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
        mean = (case["nmax"] - case["nmin"]) / (hi - lo)
        mean2 = (case["nmax"] ** 2 - case["nmin"] ** 2) / (2.0 * (hi - lo))
        n, pairs = case["nsys"] * mean, case["nsys"] * mean2 * case["steps"]
    elif kind == "planets":
        massive = 1 + case["nplanets"]
        n = case["nsys"] * (massive + case["ntest"])
        pairs = n * massive * case["steps"]
    elif kind == "probes":
        n, pairs = case["n"], case["n"] * case["npts"]
        return {"bytes": 32.0 * n + 48.0 * case["npts"], "flops": FLOPS_PER_PAIR * pairs}
    elif kind == "adaptive":
        # block steps between a 32nd of the run (the spheres' centres) and a
        # quarter of it (their outskirts): each body's force about 16 times
        n, pairs = case["n"], 16.0 * case["n"] ** 2
    else:
        n, pairs = case["n"], float(case["n"]) ** 2 * case.get("steps", 1)
        if kind in ("force", "potential", "device"):
            return {"bytes": (32.0 + {"force": 24, "potential": 8, "device": 32}[kind]) * n,
                    "flops": FLOPS_PER_PAIR * pairs}
    return {"bytes": 104.0 * n, "flops": FLOPS_PER_PAIR * pairs}


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _sums(tx, sx, sm, h, chunk=1 << 25, acc=True, pot=False):
    """Softened accelerations and potentials (Gadget-2 cubic spline) at tx from the sources."""
    a = torch.zeros_like(tx)
    p = torch.zeros(tx.shape[0], dtype=tx.dtype, device=tx.device)
    src = sx.T.contiguous()
    step = max(1, chunk // max(1, sx.shape[0]))
    for i in range(0, tx.shape[0], step):
        d = [src[k][None, :] - tx[i:i + step, k, None] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        near = torch.nonzero(((r2 < h * h) & (r2 > 0)).flatten()).flatten()   # few
        inv = torch.where(r2 > 0, r2, math.inf).rsqrt()
        f = inv * inv * inv
        q = inv
        if near.numel():
            u = r2.flatten()[near].sqrt() / h
            u2 = u * u
            inner = 10.666666666667 + u2 * (32.0 * u - 38.4)
            outer = 21.333333333333 - 48.0 * u + 38.4 * u2 - 10.666666666667 * u2 * u - 0.066666666667 / (u2 * u)
            f.view(-1)[near] = torch.where(u < 0.5, inner, outer) / h ** 3
            win = -2.8 + u2 * (5.333333333333 + u2 * (6.4 * u - 9.6))
            wout = -3.2 + 0.066666666667 / u + u2 * (10.666666666667 + u * (-16.0 + u * (9.6 - 2.133333333333 * u)))
            q.view(-1)[near] = -torch.where(u < 0.5, win, wout) / h
        if acc:
            f = f * sm
            for k in range(3):
                a[i:i + step, k] = (f * d[k]).sum(1)
        if pot:
            p[i:i + step] = -(q * sm).sum(1)
    return a, p


def _kdk(pos, vel, force, dt, steps):
    """The half kick of prepare() and the steps of run()."""
    vel = vel + force(pos) * (0.5 * dt)
    t = 0.0
    for _ in range(steps):
        pos = pos + vel * ((t + dt) - t)
        t = t + dt
        vel = vel + force(pos) * dt
    return pos, vel


def exact(case, seed):
    kind = case["kind"]
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")

    def to(v):
        return torch.from_numpy(np.ascontiguousarray(v)).to(dev)

    if kind == "adaptive" or (kind == "collision" and case["n"] > 200000):
        return None   # no closed list of steps; or too long
    if kind == "clusters":
        off, pos, vel, mass, h = _clusters(case, seed)
        out_p, out_v = [], []
        for s in range(case["nsys"]):
            sl = slice(int(off[s]), int(off[s + 1]))
            x, v, m = to(pos[sl]), to(vel[sl]), to(mass[sl])
            x, v = _kdk(x, v, lambda y: _sums(y, y, m, float(h[s]))[0], DT[kind], case["steps"])
            out_p.append(x)
            out_v.append(v)
        return [torch.cat(out_p), torch.cat(out_v)]
    if kind == "planets":
        p = _planets(case, seed)
        per, nm, ns = p["per_system"], 1 + case["nplanets"], case["nsys"]
        x, v = to(p["pos"]).reshape(ns, per, 3), to(p["vel"]).reshape(ns, per, 3)
        m = to(p["mass"]).reshape(ns, per)[:, :nm]
        dt, self_pair = DT[kind], torch.zeros((per, nm), dtype=torch.bool, device=dev)
        for k in range(nm):
            self_pair[k, k] = True

        def force(y):
            d = y[:, None, :nm, :] - y[:, :, None, :]
            r2 = (d * d).sum(-1).masked_fill(self_pair, math.inf)
            return (d * (m[:, None, :] * r2 ** -1.5)[..., None]).sum(2)

        a = force(x)
        v = v + a * (0.5 * dt)
        t, energies = 0.0, []
        for k in range(1, case["steps"] + 1):
            x = x + v * ((t + dt) - t)
            t = t + dt
            a = force(x)
            v = v + a * dt
            if k % case["every"] == 0:
                w = (v - 0.5 * dt * a)[:, :nm]
                d = x[:, None, :nm, :] - x[:, :nm, None, :]
                r = (d * d).sum(-1).masked_fill(self_pair[:nm], math.inf).sqrt()
                energies.append(0.5 * (m * (w * w).sum(-1)).sum(1)
                                - 0.5 * (m[:, :, None] * m[:, None, :] / r).sum((1, 2)))
        return [torch.stack(energies, dim=1), x.reshape(-1, 3), v.reshape(-1, 3)]
    pos, vel, mass = _system(case, seed)
    x, v, m, h = to(pos), to(vel), to(mass), case["h"]
    if case["mode"] == "fp32":   # the state the caller asked for
        x, v, m = x.float().double(), v.float().double(), m.float().double()
    if kind in ("steps", "collision", "disc"):
        x, v = _kdk(x, v, lambda y: _sums(y, y, m, h)[0], DT[kind], case["steps"])
        return [x, v]
    if kind == "force":
        return [_sums(x, x, m, h)[0]]
    if kind == "potential":
        return [_sums(x, x, m, h, acc=False, pot=True)[1]]
    if kind == "probes":
        pts = to(_points(case, seed))
        if case["mode"] == "fp32":
            pts = pts.float().double()
        return [_sums(pts, x, m, h)[0]]
    a, p = _sums(x, x, m, h, pot=True)
    return [torch.cat([a.T, p[None, :]]).contiguous()]
