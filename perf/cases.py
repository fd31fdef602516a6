"""Workloads of the framework, one pass each, for timing and for comparing results.

A case is a dict of plain values with a "kind":

  run      a whole aggregation run as `mcac_run` or a script does it: a
           Simulation is made from a parameter text, runs to its stop criterion
           (or a step cap) and its aggregates and spheres are read.  The
           parameter texts are those of tests/configs (lognormal and normal
           monomers of 30 nm, with and without an overlap correction, with
           surface growth) at their sizes and below.
  resume   a resident Simulation of a large box carries on by a number of MC
           steps and its spheres are read: one interval of a long run (the
           N = 1e6 box is the framework's headline benchmark).
  batch    an ensemble of small boxes on one GPU (mcac_amd.ensemble), grouped
           launches or one box per worker.
  search   contact searches of a caller that drives a Box through its own loop:
           monomers (the smallest call) or aggregates of many spheres.
  step     one whole collision through the Box calls: state uploaded, move to
           contact, merge, geometry and members read back.
  grow     one surface-growth update of every aggregate of a resident box.

Lengths are in metres.
"""
import ctypes
import math

import numpy as np

import mcac_amd
from mcac_amd import ensemble

DIAMETER = 30.0       # nm, the monomers of every parameter file
SIGMA = 1.25          # geometric standard deviation of the lognormal ones
N_DIV = 10            # Verlet divisions of every parameter file


def listed():
    return [
        # the smallest whole run of the ensemble list: launches and latency count
        dict(name="run_500", kind="run", n=500, fv=2e-3, temperature=1500.0, mode="normal", method="none", flux=0.0,
             stop=50, steps=0),
        # a box of the serving list, odd size
        dict(name="run_2347", kind="run", n=2347, fv=4e-3, temperature=1700.0, mode="lognormal", method="none",
             flux=0.0, stop=234, steps=0),
        # dense box run on until few, large aggregates are left: large movers, large merges
        dict(name="run_dense_6000", kind="run", n=6000, fv=0.05, temperature=1700.0, mode="lognormal", method="none",
             flux=0.0, stop=40, steps=0),
        # overlap correction by spherical caps
        dict(name="run_caps_3000", kind="run", n=3000, fv=0.05, temperature=1700.0, mode="lognormal", method="caps",
             flux=0.0, stop=300, steps=0),
        # surface growth: every step updates every aggregate
        dict(name="run_growth_2000", kind="run", n=2000, fv=1e-3, temperature=1700.0, mode="lognormal", method="none",
             flux=1e-3, stop=200, steps=3000),
        # an ensemble box at the upper end of the list, mid-run intervals
        dict(name="resume_50k", kind="resume", n=50000, fv=2e-3, temperature=1500.0, mode="normal", steps=5000),
        # the headline box
        dict(name="resume_1m", kind="resume", n=1000000, fv=3e-3, temperature=1700.0, mode="lognormal", steps=5000),
        # ensemble of small boxes in grouped launches
        dict(name="batch_64", kind="batch", boxes=64, n_min=500, n_max=5000, workers=8, group=8, depth=8, steps=4000),
        # single searches of a small monomer box: call latency
        dict(name="search_1000x1", kind="search", aggs=1000, size=1, calls=64),
        # searches among aggregates as late in a long run
        dict(name="search_2000x100", kind="search", aggs=2000, size=100, calls=64),
        # one collision of two large aggregates from a saved state
        dict(name="step_125x700", kind="step", aggs=125, size=700),
        # growth of a large resident box
        dict(name="grow_100000x8", kind="grow", aggs=100000, size=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "resume", "batch", "search", "search", "step", "grow"])
    if kind == "run":
        method = rng.choice(["none", "none", "none", "caps", "alphas", "arvo"])
        flux = rng.choice([0.0, 0.0, 1e-3, 30.0]) if method == "none" else 0.0
        n = _log(rng, 500, 1500 if method != "none" or flux else 4000)
        return dict(kind=kind, n=n, fv=math.exp(rng.uniform(math.log(2e-3), math.log(0.05))),
                    temperature=rng.uniform(1000.0, 2000.0), mode=rng.choice(["normal", "lognormal"]), method=method,
                    flux=flux, stop=max(30, n // rng.choice([5, 10, 40])), steps=1500 if flux else 30000)
    if kind == "resume":
        return dict(kind=kind, n=_log(rng, 30000, 400000), fv=rng.uniform(1e-3, 5e-3),
                    temperature=rng.uniform(1000.0, 2000.0), mode=rng.choice(["normal", "lognormal"]),
                    steps=rng.randrange(2000, 4000))
    if kind == "batch":
        return dict(kind=kind, boxes=rng.randrange(8, 48), n_min=500, n_max=_log(rng, 800, 5000), workers=8,
                    group=rng.choice([0, 4, 8]), depth=rng.choice([4, 8]), steps=rng.randrange(1000, 3000))
    if kind == "search":
        aggs = _log(rng, 200, 20000)
        return dict(kind=kind, aggs=aggs, size=_log(rng, 1, max(2, min(400, 400000 // aggs))),
                    calls=rng.randrange(16, 64))
    if kind == "step":
        return dict(kind=kind, aggs=rng.choice([8, 27, 64, 125]), size=_log(rng, 3, 700))
    aggs = _log(rng, 200, 100000)
    return dict(kind=kind, aggs=aggs, size=_log(rng, 1, max(2, min(300, 800000 // aggs))))


# ---- parameter files -------------------------------------------------------

def _ini(case, seed):
    text = ensemble.box_ini(case["n"], case["fv"], case["temperature"], seed, mean_d=DIAMETER,
                            sd_d=3.0 if case["mode"] == "normal" else SIGMA, mode=case["mode"],
                            growth_flux=case.get("flux", 0.0))
    if case.get("stop"):
        text = text.replace(f"number_of_aggregates = {max(1, int(case['n'] * 0.1))}",
                            f"number_of_aggregates = {case['stop']}")
    if case.get("method", "none") != "none":
        text += f"\n[surface_growth]\nvolsurf_method = {case['method']}\n"
    return text


def _batch_inis(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for b in range(case["boxes"]):
        n = int(round(math.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"])))))
        out.append(ensemble.box_ini(n, float(rng.uniform(1e-4, 5e-3)), float(rng.uniform(1000, 2000)),
                                    1000 + seed % 100000 + b))
    return out


# ---- boxes of synthetic aggregates ----------------------------------------

def _state(case, seed):
    """A box of `aggs` chain-like aggregates of about `size` touching spheres
    on a jittered lattice, none touching another: spheres, aggregates, the box
    side and the largest rmax."""
    rng = np.random.default_rng([seed, case["aggs"], case["size"]])
    A, mean = case["aggs"], case["size"]
    lo, hi = max(1, mean // 2 + mean % 2), mean + mean // 2
    cnt = rng.integers(lo, hi + 1, A) if mean > 1 and case["kind"] != "step" else np.full(A, mean, np.int64)
    first = np.concatenate([[0], np.cumsum(cnt)[:-1]])
    S = int(cnt.sum())
    owner = np.repeat(np.arange(A), cnt)
    r = 0.5e-9 * DIAMETER * np.exp(math.log(SIGMA) * rng.normal(size=S).clip(-3, 3))
    rel = np.zeros((S, 3))
    way = rng.normal(size=(A, 3))
    way /= np.linalg.norm(way, axis=1)[:, None]
    for k in range(1, int(cnt.max())):  # sphere k touches sphere k - 1
        on = np.nonzero(cnt > k)[0]
        way[on] += 0.8 * rng.normal(size=(len(on), 3))
        way[on] /= np.linalg.norm(way[on], axis=1)[:, None]
        i = first[on] + k
        rel[i] = rel[i - 1] + (r[i] + r[i - 1])[:, None] * way[on]
    vol, surf = 4.0 / 3.0 * math.pi * r ** 3, 4.0 * math.pi * r ** 2
    volume, surface = np.add.reduceat(vol, first), np.add.reduceat(surf, first)
    rcm = np.add.reduceat(vol[:, None] * rel, first) / volume[:, None]
    dist = np.linalg.norm(rel - rcm[owner], axis=1)
    rmax = np.maximum.reduceat(dist + r, first)
    m = math.ceil(A ** (1.0 / 3.0) - 1e-9)
    pitch = 2.3 * float(rmax.max())
    L = m * pitch
    site = rng.permutation(m ** 3)[:A]
    cell = np.stack([site // (m * m), site // m % m, site % m], axis=1)
    slack = (0.5 * pitch - rmax)[:, None]
    pos = (cell + 0.5) * pitch + rng.uniform(-0.95, 0.95, (A, 3)) * slack
    xyz = (pos - rcm)[owner] + rel
    spheres = dict(x=xyz[:, 0].copy(), y=xyz[:, 1].copy(), z=xyz[:, 2].copy(), r=r, vol=vol, surf=surf,
                   rx=rel[:, 0].copy(), ry=rel[:, 1].copy(), rz=rel[:, 2].copy())
    aggs = dict(pos=pos, rcm=rcm, rmax=rmax, volume=volume, surface=surface, count=cnt.astype(np.int64),
                members=np.arange(S, dtype=np.int64))
    return spheres, aggs, first, L, float(rmax.max()), pitch, rng


def _searches(case, seed):
    spheres, aggs, first, L, rmax, pitch, rng = _state(case, seed)
    movers = rng.integers(0, case["aggs"], case["calls"])
    dirs = rng.normal(size=(case["calls"], 3))
    dirs /= np.linalg.norm(dirs, axis=1)[:, None]
    lpms = rng.uniform(0.3, 2.5, case["calls"]) * pitch
    return spheres, aggs, first, L, rmax, movers, dirs, lpms


def _collision(case, seed):
    """The state, and a move of one aggregate that brings it onto another: a
    sphere of the mover heads for a sphere of its target."""
    spheres, aggs, first, L, rmax, pitch, rng = _state(case, seed)
    mover, target = (int(v) for v in rng.permutation(case["aggs"])[:2])
    i = int(first[mover] + rng.integers(aggs["count"][mover]))
    j = int(first[target] + rng.integers(aggs["count"][target]))
    d = np.array([spheres[k][j] - spheres[k][i] for k in "xyz"])
    d -= L * np.round(d / L)
    gap = float(np.linalg.norm(d))
    return spheres, aggs, first, L, rmax, mover, d / gap, gap


def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        return dict(case=case, ini=_ini(case, seed))
    if kind == "resume":
        return dict(case=case, sim=mcac_amd.Simulation(_ini(case, seed)))
    if kind == "batch":
        return dict(case=case, inis=_batch_inis(case, seed))
    if kind == "step":
        spheres, aggs, _, L, rmax, mover, direction, lpm = _collision(case, seed)
        box = mcac_amd.Box(L, N_DIV, len(spheres["x"]), case["aggs"])
        return dict(case=case, box=box, spheres=spheres, aggs=aggs, mover=mover, dir=direction, lpm=lpm, rmax=rmax)
    if kind == "search":
        spheres, aggs, _, L, rmax, movers, dirs, lpms = _searches(case, seed)
        box = mcac_amd.Box(L, N_DIV, len(spheres["x"]), case["aggs"])
        box.upload(spheres, aggs)
        return dict(case=case, box=box, movers=[int(m) for m in movers], dirs=dirs, lpms=[float(v) for v in lpms],
                    rmax=rmax)
    spheres, aggs, _, L, rmax, _, _ = _state(case, seed)
    box = mcac_amd.Box(L, N_DIV, len(spheres["x"]), case["aggs"])
    box.upload(spheres, aggs)
    return dict(case=case, box=box, out=[np.zeros(case["aggs"]) for _ in range(5)])


def _by_id(aggs, n):
    """The live aggregates' values at their ids, 0 elsewhere (a run's records are kept so)."""
    out = {}
    for k, v in aggs.items():
        if k != "uid":
            out[k] = np.zeros(n, v.dtype)
            out[k][aggs["uid"]] = v
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        sim = mcac_amd.Simulation(state["ini"])
        steps = sim.run(case["steps"]) if case["steps"] else sim.run()
        out = dict(steps=steps, time=sim.scalar("time"), aggregates=_by_id(sim.aggregates(), case["n"]),
                   spheres=sim.box().spheres())
        sim.close()
        return out
    if kind == "resume":
        sim = state["sim"]
        steps = sim.run(case["steps"])
        return dict(steps=steps, time=sim.scalar("time"), n_agg=int(sim.scalar("n_agg")), spheres=sim.box().spheres())
    if kind == "batch":
        out = ensemble.batch_run(state["inis"], workers=case["workers"], max_steps=case["steps"],
                                 boxes_per_worker=case["group"], depth=case["depth"])
        return {k: out[k] for k in ("steps", "status", "final_time") if k in out}
    if kind == "search":
        box, rmax = state["box"], state["rmax"]
        found = [box.next_contact(m, d, l, rmax) for m, d, l in zip(state["movers"], state["dirs"], state["lpms"])]
        found = np.array(found)
        return {k: found[k] for k in ("distance", "moving_sphere", "other_sphere", "other_agg", "contact", "n_query",
                                      "n_filtered", "n_pairs")}
    if kind == "step":
        box = state["box"]
        box.upload(state["spheres"], state["aggs"])
        hit = box.next_contact(state["mover"], state["dir"], state["lpm"], state["rmax"], move=True)
        merged = box.merge(hit)
        aggs = box.aggregates()
        geometry = {k: merged[k] for k in ("volume", "surface", "rg", "rmax", "radius_sum", "com", "rcm",
                                           "overlapping", "coordination")}
        return dict(distance=hit["distance"], keeper=merged["keeper"], removed=merged["removed"], n=merged["n"],
                    geometry=geometry, members=box.members(int(merged["keeper"])), pos=aggs["pos"], count=aggs["count"])
    out = state["out"]
    ptr = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in out]
    dr = 1e-13  # the growth of a step of microseconds at the configurations' fluxes
    rc = mcac_amd.load_gpu().mcac_box_grow(state["box"].h, dr, *ptr)
    if rc:
        raise RuntimeError(f"mcac_box_grow: status {rc}")
    return dict(zip(("volume", "surface", "radius_sum", "rg", "rmax"), out))


# ---- what a pass cannot do without -----------------------------------------

def work(case):
    """Bytes and FP64 operations of one pass.  A step reads a 36 B row (centre,
    radius, id) of each aggregate in the 4^3 of 10^3 cells around its mover and
    about 40 operations on it, then its mover's spheres; a run of n monomers to
    n / 10 takes about 15 n steps."""
    kind = case["kind"]

    def steps_of(n, steps, agg):
        seen = max(1.0, 0.064 * agg)
        return dict(bytes=steps * (36.0 * seen + 96.0), flops=steps * 40.0 * seen)

    if kind == "run":
        n = case["n"]
        steps = min(case["steps"] or 15.0 * n, 15.0 * n)
        w = steps_of(n, steps, 0.4 * n)
        if case["flux"]:  # every sphere and aggregate of every step
            w["bytes"] += steps * 168.0 * 0.8 * n
            w["flops"] += steps * 60.0 * n
        return w
    if kind == "resume":
        w = steps_of(case["n"], case["steps"], case["n"])
        w["bytes"] += 64.0 * case["n"]
        return w
    if kind == "batch":
        mean = (case["n_max"] - case["n_min"]) / max(1e-9, math.log(case["n_max"] / case["n_min"]))
        w = steps_of(mean, case["steps"], 0.6 * mean)
        return {k: v * case["boxes"] for k, v in w.items()}
    if kind == "search":
        seen = 0.3 * case["aggs"]
        pairs = 2.0 * case["size"]
        return dict(bytes=case["calls"] * (36.0 * seen + 32.0 * 3 * case["size"]),
                    flops=case["calls"] * (40.0 * seen + 40.0 * pairs))
    S = case["aggs"] * case["size"]
    if kind == "step":
        n = 2.0 * case["size"]
        return dict(bytes=76.0 * S + 124.0 * case["aggs"] + 200.0 * n, flops=40.0 * case["aggs"] + 12.0 * n * n / 2)
    return dict(bytes=(72.0 + 72.0 + 4.0) * S + 190.0 * case["aggs"], flops=60.0 * S)


# ---- the same in plain numpy -----------------------------------------------

def _swept(p1, r1, p2, r2, d, dist, L):
    """Travel to first contact of spheres p1 (n, 3) moving along d by at most
    dist with p2 (m, 3), any periodic image: the smallest over all pairs."""
    best = math.inf
    for i in range(0, len(p1), 64):
        g = p2[None, :, :] - p1[i:i + 64, None, :]
        g -= L * np.floor(g / L)
        s = r1[i:i + 64, None] + r2[None, :]
        for shift in np.ndindex(2, 2, 2):  # the images next to the mover and ahead of it
            h = g - L * np.array(shift)
            h2 = (h * h).sum(-1)
            if (h2 <= s * s).any():
                return 0.0
            proj = h @ d
            axis = np.maximum(h2 - proj * proj, 0.0)
            reach = np.where((proj >= 0) & (axis <= s * s), proj - np.sqrt(np.maximum(s * s - axis, 0.0)), math.inf)
            best = min(best, float(reach.min()))
    return best if best <= dist else math.inf


def _first_contact(spheres, aggs, first, L, mover, d, lpm):
    xyz = np.stack([spheres[k] for k in "xyz"], axis=1)
    mine = slice(first[mover], first[mover] + aggs["count"][mover])
    g = aggs["pos"] - aggs["pos"][mover]
    g -= L * np.round(g / L)  # the sweep and the radii stay within half the box
    g -= np.clip(g @ d, 0.0, lpm)[:, None] * d
    near = np.linalg.norm(g, axis=1) <= aggs["rmax"] + aggs["rmax"][mover] + 1e-9
    near[mover] = False
    owner = np.repeat(np.arange(len(first)), aggs["count"])
    other = near[owner]
    if not other.any():
        return math.inf
    return _swept(xyz[mine], spheres["r"][mine], xyz[other], spheres["r"][other], d, lpm, L)


def exact(case, seed):
    kind = case["kind"]
    if kind == "search":
        spheres, aggs, first, L, _, movers, dirs, lpms = _searches(case, seed)
        if case["calls"] * case["size"] ** 2 * 60 > 2e8 or lpms.max() + 2 * aggs["rmax"].max() > 0.5 * L:
            return None
        dist = np.array([_first_contact(spheres, aggs, first, L, int(m), d, float(l))
                         for m, d, l in zip(movers, dirs, lpms)])
        return dict(distance=dist, moving_sphere=None, other_sphere=None, other_agg=None, contact=None, n_query=None,
                    n_filtered=None, n_pairs=None)
    if kind == "step":
        spheres, aggs, first, L, _, mover, d, lpm = _collision(case, seed)
        if lpm + 2 * aggs["rmax"].max() > 0.5 * L:
            return None
        return dict(distance=_first_contact(spheres, aggs, first, L, mover, d, lpm), keeper=None, removed=None, n=None,
                    geometry=None, members=None, pos=None, count=None)
    if kind == "grow":
        spheres, aggs, first, _, _, _, _ = _state(case, seed)
        owner = np.repeat(np.arange(case["aggs"]), aggs["count"])
        rel = np.stack([spheres[k] for k in ("rx", "ry", "rz")], axis=1)
        r = spheres["r"] + 1e-13
        vol = 4.0 / 3.0 * math.pi * r ** 3
        volume = np.add.reduceat(vol, first)
        rcm = np.add.reduceat(vol[:, None] * rel, first) / volume[:, None]
        dist = np.linalg.norm(rel - rcm[owner], axis=1)
        rg = np.sqrt(np.add.reduceat(vol * dist ** 2 + 0.6 * vol * r ** 2, first) / volume)
        return dict(volume=volume, surface=np.add.reduceat(4.0 * math.pi * r ** 2, first),
                    radius_sum=np.add.reduceat(r, first), rg=rg, rmax=np.maximum.reduceat(dist + r, first))
    return None
