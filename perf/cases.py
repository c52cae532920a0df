"""What the speed of this library is measured on.

Two ways into the library are in use.  A driver that keeps its own time loop
calls the drop-in functions of `sph_2_amd.libsx` once per step with numpy
arrays on the host (density, smoothing lengths, gravity, hydro), and a run that
stays on the device is stepped by `sph_2_amd.plan.SphPlan` on the caller's
device arrays, or packed with others in a `sph_2_amd.serve.Batch`.  The cases
take both, from a few thousand particles, where the launches and copies of a
call are most of it, to the million-particle run, with the sizes of the
reference's recorded runs, of the test suite and of the benchmark.

The particles are an Evrard sphere in collapse (rho ~ 1/r, infall plus a few
percent of noise, u and masses as the case says), a Plummer sphere or the
turbulent cooling cloud, made from the seed.
"""
import math

import numpy as np
import torch

from sph_2_amd import ic, libsx
from sph_2_amd.plan import SphPlan
from sph_2_amd.serve import Batch, default_cooling

DT = 1e-4


def listed():
    return [
        # getDensity of a small run, as a driver's loop calls it every step: copies and launches
        {"name": "density_2048", "kind": "density", "n": 2048, "masses": "equal"},
        # the smoothing lengths of one rank's particles a step later (mpi4py driver, the size of
        # the reference's recorded runs): h and counts of the step before, eq. 31 start
        {"name": "smoothing_65752", "kind": "smoothing", "n": 65752, "rule": "mpi3"},
        # the first smoothing lengths of a new set of particles, from the density profile's guess
        {"name": "h_first_16384", "kind": "smoothing", "n": 16384, "rule": "h_smooth_fast"},
        # direct-sum gravity of an ordinary run, an odd size, particles of several masses
        {"name": "gravity_20011", "kind": "gravity", "n": 20011, "masses": "varied"},
        # hydro acceleration and du/dt of a larger run with the standard viscosity
        {"name": "hydro_100003", "kind": "hydro", "n": 100003, "av_form": 0, "masses": "equal"},
        # tree gravity of a large collisionless set (Plummer sphere)
        {"name": "tree_524288", "kind": "tree", "n": 524288, "theta": 0.5},
        # resident runs, the whole step: the smallest (ten steps between two snapshots) ...
        {"name": "step_4096", "kind": "step", "n": 4096, "steps": 10, "gravity": "direct",
         "h_mode": 0, "masses": "equal"},
        # ... the size of the reference's recorded runs ...
        {"name": "step_65752", "kind": "step", "n": 65752, "steps": 2, "gravity": "direct",
         "h_mode": 0, "masses": "equal"},
        # ... and the largest: the benchmark's headline step
        {"name": "step_1048576", "kind": "step", "n": 1048576, "steps": 1, "gravity": "direct",
         "h_mode": 0, "masses": "equal"},
        # the same run with tree gravity
        {"name": "tree_step_1048576", "kind": "step", "n": 1048576, "steps": 1, "gravity": "tree",
         "h_mode": 0, "masses": "equal"},
        # the turbulent cloud with the implicit cooling solve in every step
        {"name": "cloud_131072", "kind": "cloud", "n": 131072, "steps": 2},
        # served runs of uneven size, packed, advanced together from captured graphs, copied out
        {"name": "served_8_runs", "kind": "served", "runs": 8, "n_min": 2048, "n_max": 32768,
         "steps": 10},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["density", "smoothing", "gravity", "hydro", "tree", "step", "step", "step",
                       "cloud", "served"])
    masses = rng.choice(["equal", "equal", "varied"])
    if kind == "density":
        return {"kind": kind, "n": _log_uniform(rng, 2048, 131072), "masses": masses}
    if kind == "smoothing":
        return {"kind": kind, "n": _log_uniform(rng, 2048, 131072),
                "rule": rng.choice(["mpi3", "mpi3", "h_smooth_fast", "knn"])}
    if kind == "gravity":
        return {"kind": kind, "n": _log_uniform(rng, 2048, 131072), "masses": masses}
    if kind == "hydro":
        return {"kind": kind, "n": _log_uniform(rng, 2048, 131072),
                "av_form": rng.choice([0, 1]), "masses": masses}
    if kind == "tree":
        return {"kind": kind, "n": _log_uniform(rng, 32768, 524288),
                "theta": rng.choice([0.3, 0.5, 0.5, 0.7])}
    if kind == "step":
        gravity = rng.choice(["direct", "direct", "tree"])
        h_mode = rng.choice([0, 0, 0, 2])
        top = 1048576 if h_mode == 0 and gravity == "tree" else 262144
        n = _log_uniform(rng, 2048, top)
        return {"kind": kind, "n": n, "steps": 10 if n < 16384 else 2 if n < 262144 else 1,
                "gravity": gravity, "h_mode": h_mode, "masses": masses}
    if kind == "cloud":
        return {"kind": kind, "n": _log_uniform(rng, 8192, 262144), "steps": 2}
    return {"kind": kind, "runs": rng.randint(2, 8), "n_min": 2048,
            "n_max": _log_uniform(rng, 16384, 65536), "steps": 10}


# ---------------------------------------------------------------------------
# Particles
# ---------------------------------------------------------------------------
def _rng(seed):
    return np.random.default_rng(int(seed) & 0xFFFFFFFF)


def _collapse(n, seed, masses):
    """An Evrard sphere in collapse."""
    e = ic.evrard(n, seed=int(seed))
    g = _rng(seed)
    r = np.sqrt((e.pos ** 2).sum(axis=1))
    infall = -0.8 / (0.3 + r)
    e.vel = infall[:, None] * e.pos + 0.05 * g.standard_normal((n, 3))
    e.u = 0.05 * (1.0 + 0.5 * (1.0 - r)) * g.uniform(0.95, 1.05, n)
    if masses == "varied":
        w = g.uniform(0.5, 1.5, n)
        e.m = w / w.sum()
    return e


def _gas(e, seed):
    """rho, P and c of the sphere's profile, with a few percent of noise."""
    g = _rng(seed + 1)
    r = np.sqrt((e.pos ** 2).sum(axis=1))
    rho = g.uniform(0.95, 1.05, e.n) / (2.0 * np.pi * np.maximum(r, 1e-2))
    return rho, (2.0 / 3.0) * rho * e.u, np.sqrt(10.0 / 9.0 * e.u)


def _served_sizes(case):
    """Sizes of the served runs: spread evenly in the logarithm, the largest at n_max."""
    k = case["runs"]
    f = math.log(case["n_max"] / case["n_min"])
    return [int(round(case["n_min"] * math.exp(f * (i + 1) / k))) for i in range(k)]


# ---------------------------------------------------------------------------
# State and pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "served":
        sizes = _served_sizes(case)
        bt = Batch(sum(sizes), max_runs=len(sizes), cooling=default_cooling(), graph=True)
        bt.set_gravity_symmetric(4, 1 << 30)
        ids = []
        for k, n in enumerate(sizes):
            e = (ic.turbulent_cloud(n, seed=int(seed) + k, ng=32) if k % 2 else
                 _collapse(n, int(seed) + k, "equal"))
            ids.append(bt.admit(e, DT, cooling=bool(k % 2)))
        return {"kind": kind, "batch": bt, "ids": ids, "steps": case["steps"]}
    n = case["n"]
    if kind == "cloud":
        e = ic.turbulent_cloud(n, seed=int(seed), ng=32)
        pl = SphPlan(n, cooling=default_cooling())
    elif kind == "step":
        e = _collapse(n, seed, case["masses"])
        pl = SphPlan(n, h_mode=case["h_mode"])
        if case["gravity"] == "tree":
            pl.set_gravity_bh(0.5)
    if kind in ("cloud", "step"):
        own = [torch.from_numpy(np.ascontiguousarray(a)).cuda()
               for a in (e.pos, e.vel, e.u, e.m, e.h)]
        pl.bind(*own)
        pl.init()
        return {"kind": kind, "plan": pl, "own": own, "steps": case["steps"],
                "cooling": kind == "cloud"}
    if kind == "tree":
        e = ic.plummer(n, seed=int(seed))
        return {"kind": kind, "pos": e.pos, "m": e.m, "eps": 0.01, "theta": case["theta"]}
    e = _collapse(n, seed, case.get("masses", "equal"))
    s = {"kind": kind, "pos": e.pos, "m": e.m, "h": e.h}
    if kind == "smoothing":
        s["rule"] = case["rule"]
        if case["rule"] == "mpi3":
            # the particles have drifted for a long step since h and k were found
            h, k, _ = libsx.smoothing_h(e.pos, e.h)
            r = np.sqrt((e.pos ** 2).sum(axis=1))
            s.update(h=h, k=k, pos=e.pos + 1e-3 * e.vel, dt=1e-3,
                     divv=-0.8 * (0.9 + 2.0 * r) / (0.3 + r) ** 2)
    elif kind == "hydro":
        s["rho"], s["P"], s["c"] = _gas(e, seed)
        s["vel"], s["av_form"] = e.vel, case["av_form"]
    return s


def run(s):
    kind = s["kind"]
    if kind == "density":
        return libsx.getDensity(s["pos"], s["m"], s["h"])
    if kind == "smoothing":
        if s["rule"] == "mpi3":
            return libsx.smoothing_fast_new_mpi3(0, len(s["h"]), s["pos"], s["h"], s["k"],
                                                 s["divv"], s["dt"])
        if s["rule"] == "knn":
            return libsx.do_smoothingX((s["pos"], s["pos"]))
        return libsx.h_smooth_fast(s["pos"], s["h"])
    if kind == "gravity":
        return libsx.getAcc_g_smth(s["pos"], s["m"], 1.0, s["h"])
    if kind == "hydro":
        return libsx.getAcc_sph_dU(s["pos"], s["vel"], s["rho"], s["P"], s["c"], s["h"], s["m"],
                                   av_form=s["av_form"])
    if kind == "tree":
        return libsx.getAcc_g_bh(s["pos"], s["m"], 1.0, s["eps"], s["theta"])
    if kind == "served":
        s["batch"].step(s["steps"])
        out = [s["batch"].store(i) for i in s["ids"]]
        return [{f: o[f] for f in ("pos", "vel", "u", "h", "k")} for o in out]
    s["plan"].step(s["steps"], DT, cooling=s["cooling"])
    pos, vel, u, _, h = s["own"]
    return {"pos": pos, "vel": vel, "u": u, "h": h}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
PAIR = 24    # flop of one gravity pair applied to both particles (r^2, r^-3, two force sums)
NGB = 64     # neighbours of a particle


def _step_work(n, gravity):
    # density and EOS, div/curl and hydro over the neighbours; gravity
    flops = n * NGB * (20 + 30 + 50)
    flops += PAIR * n * (n - 1) / 2 if gravity == "direct" else 20 * n * 40 * math.log2(n)
    # pos, vel, u, h in and out, m and du/dt of the step before in, du/dt out
    return {"bytes": 8.0 * n * (2 * 8 + 3), "flops": float(flops)}


def work(case):
    kind = case["kind"]
    if kind == "served":
        w = [_step_work(n, "direct") for n in _served_sizes(case)]
        return {k: case["steps"] * sum(x[k] for x in w) for k in ("bytes", "flops")}
    n = case["n"]
    if kind in ("step", "cloud"):
        w = _step_work(n, case.get("gravity", "direct"))
        return {k: case["steps"] * w[k] for k in w}
    if kind == "density":
        return {"bytes": 8.0 * n * 6, "flops": 20.0 * n * NGB}
    if kind == "smoothing":
        return {"bytes": 8.0 * n * 5 + 8.0 * n, "flops": 8.0 * n * NGB}
    if kind == "gravity":
        return {"bytes": 8.0 * n * 8, "flops": PAIR * n * (n - 1) / 2.0}
    if kind == "hydro":
        return {"bytes": 8.0 * n * 15, "flops": 50.0 * n * NGB}
    return {"bytes": 8.0 * n * 8, "flops": 20.0 * n * 40 * math.log2(n)}


# ---------------------------------------------------------------------------
# The same values in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _close_pairs(x, reach, rows=None):
    """Index pairs (i, j) of each chunk of rows with |x_i - x_j| <= reach(i, j)
    and their exact separations."""
    n = len(x)
    step = max(1, int(1.5e8 // n))
    sq = (x * x).sum(1)
    for a in range(0, n, step):
        b = min(n, a + step)
        r2 = torch.addmm(sq[None, :] + sq[a:b, None], x[a:b], x.T, alpha=-2.0)
        t = reach(a, b)
        i, j = torch.nonzero(r2 <= t * t * (1.0 + 1e-9) + 1e-12, as_tuple=True)
        i = i + a
        d = x[i] - x[j]
        r2 = (d[:, 0] ** 2 + d[:, 1] ** 2) + d[:, 2] ** 2
        yield i, j, d, r2


def _density64(s):
    x, m, h = _dev(s["pos"]), _dev(s["m"]), _dev(s["h"])
    rho = torch.zeros_like(m)
    for i, j, _, r2 in _close_pairs(x, lambda a, b: h[a:b, None] + h[None, :]):
        t = h[i] + h[j]
        q = torch.sqrt(r2) / (0.5 * t)
        w = torch.where(q <= 1.0, 1.0 - 1.5 * q ** 2 + 0.75 * q ** 3,
                        0.25 * (2.0 - q).clamp(min=0.0) ** 3) / (math.pi * (0.5 * t) ** 3)
        rho.index_add_(0, i, torch.where(r2 <= t * t, m[j] * w, torch.zeros_like(w)))
    return rho.cpu().numpy()


def _hydro64(s):
    x, v = _dev(s["pos"]), _dev(s["vel"])
    rho, P, c, h, m = (_dev(s[k]) for k in ("rho", "P", "c", "h", "m"))
    pr = P / rho ** 2
    acc, du = torch.zeros_like(x), torch.zeros_like(m)
    for i, j, d, r2 in _close_pairs(x, lambda a, b: h[a:b, None] + h[None, :]):
        keep = (r2 <= (h[i] + h[j]) ** 2) & (i != j)
        i, j, d, r2 = i[keep], j[keep], d[keep], r2[keep]
        hij = 0.5 * (h[i] + h[j])
        r = torch.sqrt(r2)
        q = r / hij
        F = torch.where(q <= 1.0, -3.0 + 2.25 * q, -0.75 * (2.0 - q) ** 2 / q) / (math.pi * hij ** 5)
        vr = ((v[i] - v[j]) * d).sum(1)
        rhob = 0.5 * (rho[i] + rho[j])
        if s["av_form"] == 0:
            mu = hij * vr / (r2 + 0.01 * hij ** 2)
            pi = (-0.5 * (c[i] + c[j]) * mu + 2.0 * mu ** 2) / rhob
        else:
            w = vr / (r + 1e-5)
            pi = -0.5 * (c[i] + c[j] - 3.0 * w) * w / rhob
        pi = torch.where(vr <= 0.0, pi, torch.zeros_like(pi))
        acc.index_add_(0, i, -(m[j] * (pr[i] + pr[j] + pi) * F)[:, None] * d)
        du.index_add_(0, i, m[j] * (pr[i] + 0.5 * pi) * F * vr)
    return acc.cpu().numpy(), du.cpu().numpy()


def _gravity64(pos, m, eps):
    """Spline-softened direct sum: the point masses of all pairs beyond the
    largest softening reach in one product, the closer pairs one by one."""
    x, m, e = _dev(pos), _dev(m), _dev(np.broadcast_to(np.asarray(eps, np.float64), (len(pos),)))
    n = len(x)
    step = max(1, int(2.5e8 // n))
    sq = (x * x).sum(1)
    y = torch.cat([m[:, None] * x, m[:, None]], 1)
    reach2 = float((2.0 * e.max()) ** 2) * (1.0 + 1e-6) + 1e-12
    acc = torch.empty_like(x)
    for a in range(0, n, step):
        b = min(n, a + step)
        r2 = torch.addmm(sq[None, :] + sq[a:b, None], x[a:b], x.T, alpha=-2.0)
        near = r2 <= reach2
        i, j = torch.nonzero(near, as_tuple=True)
        r2.masked_fill_(near, float("inf"))
        r2.rsqrt_()
        w = (r2 * r2).mul_(r2) @ y
        acc[a:b] = w[:, :3] - x[a:b] * w[:, 3:]
        del r2, near
        i = i + a
        k = i != j
        i, j = i[k], j[k]
        d = x[j] - x[i]
        r = torch.sqrt((d * d).sum(1))
        ee = 0.5 * (e[i] + e[j])
        q = r / ee
        f_in = (4.0 / 3.0 - 1.2 * q ** 2 + 0.5 * q ** 3) / ee ** 3
        f_mid = (-1.0 / 15.0 + 8.0 / 3.0 * q ** 3 - 3.0 * q ** 4 + 1.2 * q ** 5 - q ** 6 / 6.0) / r ** 3
        f = torch.where(q <= 1.0, f_in, torch.where(q <= 2.0, f_mid, r ** -3))
        acc.index_add_(0, i, (m[j] * f)[:, None] * d)
    return acc.cpu().numpy()


def _knn64(pos, kth=64):
    x = _dev(pos)
    n = len(x)
    step = max(1, int(1.5e8 // n))
    out = []
    for a in range(0, n, step):
        xa = x[a:a + step]
        r2 = torch.zeros((len(xa), n), dtype=x.dtype, device=x.device)
        for c in range(3):
            d = xa[:, c, None] - x[None, :, c]
            r2 += d * d
        out.append(0.5 * torch.sqrt(torch.topk(r2, kth + 1, dim=1, largest=False)[0].max(1)[0]))
    return torch.cat(out).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "cloud", "served") or (kind == "smoothing" and case["rule"] != "knn"):
        # a whole step's state, and lengths that are where an iteration stopped
        return None
    s = prepare(case, seed)
    if kind == "density":
        return _density64(s)
    if kind == "smoothing":
        return _knn64(s["pos"])
    if kind == "hydro":
        return _hydro64(s)
    return _gravity64(s["pos"], s["m"], s["eps"] if kind == "tree" else s["h"])
