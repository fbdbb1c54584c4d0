"""The work that users of this framework have it do, as cases to be timed.

Every case runs through the public entry points (`particulator_hip`), on populations of the
sizes and settings of the repository's own configurations (the swarm, avalanche, sweep and
beam workloads of bench.py, the fields and callbacks of the tests).  A pass is one sample:
fresh initial particles on the device, the steps, and what such a program reads at the end
(whole populations where they are small enough to be brought to the host, else the
statistics, collision counters, depth dose and tallies that the run is made for)."""
import math
import os
import sys

import numpy as np
import torch  # noqa: F401  (loads the HIP runtime that the library shares)

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "particulator.jl_amd"))

import particulator_hip as P  # noqa: E402
from particulator_hip import air, co  # noqa: E402
from particulator_hip.continuum import air_loss  # noqa: E402
from particulator_hip.population import STATE_DTYPE  # noqa: E402

CUT = 1e4 * co.eV
DT = 1e-12
EMPTY = np.zeros(0, dtype=STATE_DTYPE)
_tables = {}


def _population(name, **kw):
    """A population run: n electrons in `nswarm` swarms (split evenly), E log-spaced over
    elo..ehi, energy e1 (or log-uniform e1..e2), `tracked` photons and positrons or not."""
    c = dict(family="population", name=name, nswarm=1, elo=1e6, ehi=1e6, e1=1e6, e2=0.0, all_tracked=False, mode="run",
             compact=8, roulette=0, field="homogeneous", state=False, ragged=False, capacity=0)
    c.update(kw)
    return c


def listed():
    return [
        # run! with callbacks asking for the population every step, at the smallest swarm of
        # the sweep: each step is one call and its answer (latency and launches)
        _population("loop_1e3", n=1000, steps=16, mode="loop", compact=1, state=True),
        # the runaway swarm, 10^4 electrons at 1 MeV, photons tallied, compaction each step
        _population("swarm_1e4", n=10_000, steps=200, compact=1, state=True),
        # its 32 independent samples as 32 swarms of one population
        _population("swarms_32x1e4", n=320_000, steps=200, nswarm=32),
        # a small coupled avalanche of odd size, all species followed and brought back
        _population("avalanche_40961", n=40_961, steps=200, e1=1e5, e2=1e7, all_tracked=True, state=True),
        # the coupled avalanche at a tenth of its size and at its full size
        _population("avalanche_1e6", n=1_000_003, steps=48, e1=1e5, e2=1e7, all_tracked=True),
        _population("avalanche_1e7", n=10_000_000, steps=24, e1=1e5, e2=1e7, all_tracked=True, capacity=1 << 27),
        # the field sweep: 256 uneven swarms at 0.4-4 MV/m, captured-graph replays
        _population("sweep_256", n=118_000_000, steps=16, nswarm=256, elo=0.4e6, ehi=4e6, mode="graph", ragged=True),
        # electrons crossing a double layer with a magnetic field and continuum losses (the
        # field functors and the combined forcing of the reference's scripts)
        _population("layer_1e5", n=100_003, steps=64, e1=1e5, e2=1e7, field="layer"),
        # run! with the population held by Russian roulette every step
        _population("roulette_2e5", n=200_001, steps=24, elo=4e6, ehi=4e6, mode="loop", compact=1, roulette=150_000),
        # photon pencil beam with depth dose and photon births: a reduced one over more
        # steps (electrons dominate), and the full one
        dict(family="beam", name="beam_2e6", n=2_000_000, steps=10),
        dict(family="beam", name="beam_1e8", n=100_000_000, steps=3),
        # what onoutput reads: population and per-swarm statistics of a large population
        dict(family="statistics", name="statistics_2e6", n=2_000_003, nswarm=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "run", "run", "avalanche", "avalanche", "graph", "layer", "roulette", "beam", "statistics"])
    if kind == "beam":
        n = _log(rng, 1e5, 5e7)
        c = dict(family="beam", n=n, steps=rng.randint(1, max(1, min(10, int(6e7 / n)))))
    elif kind == "statistics":
        c = dict(family="statistics", n=_log(rng, 1e4, 3e6), nswarm=rng.randint(1, 256))
    elif kind == "loop":
        c = _population("", n=_log(rng, 1e3, 3e4), steps=rng.randint(8, 40), mode="loop", compact=1, state=True)
    elif kind == "roulette":
        n = _log(rng, 1e4, 1e6)
        c = _population("", n=n, steps=rng.randint(8, 32), elo=4e6, ehi=4e6, mode="loop", compact=1,
                        roulette=int(n * rng.uniform(0.5, 1.0)))
    elif kind == "layer":
        n = _log(rng, 3e3, 1e6)
        c = _population("", n=n, steps=rng.randint(16, 128), e1=1e5, e2=1e7, field="layer", state=n <= 50_000)
    elif kind == "avalanche":
        n = _log(rng, 1e4, 1e7)
        c = _population("", n=n, steps=rng.randint(8, max(8, min(200, int(2e8 / n)))), e1=1e5, e2=1e7, all_tracked=True,
                        state=n <= 50_000, compact=rng.choice([2, 4, 8, 16]))
    elif kind == "run":
        n = _log(rng, 1e3, 3e6)
        c = _population("", n=n, steps=rng.randint(16, max(16, min(300, int(2e8 / n)))), nswarm=rng.randint(1, 32),
                        compact=rng.choice([1, 8, 8]), state=n <= 50_000)
    else:
        n = _log(rng, 3e4, 2e7)
        c = _population("", n=n, steps=rng.randint(8, max(8, min(100, int(2e8 / n)))), nswarm=rng.randint(2, 256),
                        elo=0.4e6, ehi=4e6, mode="graph", ragged=True, compact=rng.choice([4, 8]))
    c.pop("name", None)
    return c


def _fields(c):
    ns = c["nswarm"]
    return [c["elo"] * (c["ehi"] / c["elo"]) ** (i / max(1, ns - 1)) for i in range(ns)]


def _air(c):
    """tables of air, as a program builds them once for its fields"""
    key = (c.get("nswarm", 1), c.get("elo", 1e6), c.get("ehi", 1e6))
    if key not in _tables:
        if key[0] == 1:
            _tables[key] = air.build_tables(air.composition(), key[1], DT, CUT)
        else:
            _tables[key] = air.swarm_tables(air.composition(), _fields(c), DT, CUT)
    return _tables[key]


def _prepare_population(c, seed):
    te, tg, tp = _air(c)
    n, ns, al = c["n"], c["nswarm"], c["all_tracked"]
    cap = c["capacity"] or max(1 << 16, 2 * n)
    mp = P.MultiPopulation(seed=seed, nswarm=ns, tally_tracked=al, electron=P.Population(cap, [], te, CUT),
                           photon=P.Population(cap, [], tg, CUT, tracked=al),
                           positron=P.Population(cap, [], tp, CUT, tracked=al))
    if c["field"] == "layer":
        field = P.ElectromagneticField(P.DoubleLayerField(-1e-2, 1e-2, (0.0, 0.0, -2e6)),
                                       P.HomogeneousField((0.0, 5e-5, 0.0)))
        pushers = [P.RK2Pusher(P.CombinedForcing(field, air_loss(air.composition(), CUT, n=5)))]
    else:
        pushers = [P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, -e)))) for e in _fields(c)]
    for i, p in enumerate(pushers):
        mp.set_pusher(p, swarm=i)
    if c["ragged"]:  # uneven swarms, U{1e3..1e6} of the sweep scaled to n
        u = np.random.default_rng(seed).integers(1000, 1_000_001, size=ns)
        counts = np.maximum(1, (u * (n / u.sum())).astype(np.int64))
    else:
        counts = np.full(ns, n // ns, dtype=np.int64)
        counts[: n % ns] += 1
    mp.set_launch(**dict(mp.get_launch(), compact_every=c["compact"]))
    return dict(c=c, mp=mp, pusher=pushers[0], counts=[int(v) for v in counts],
                species=[0, 1, 2] if al else [0])


def _prepare_beam(c, seed):
    te, tg, tp = _air(c)
    n = c["n"]
    caps = (max(1 << 16, n // 10), int(1.1 * n) + 1024, max(1 << 15, n // 20))
    mp = P.MultiPopulation(seed=seed, tally_bins=512, tally_range=(1e4 * co.eV, 1e7 * co.eV), dose=(300, 0.0, 3.0),
                           tally_tracked=True, electron=P.Population(caps[0], [], te, CUT),
                           photon=P.Population(caps[1], [], tg, CUT), positron=P.Population(caps[2], [], tp, CUT))
    mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, 0.0)))))
    # long steps: secondaries of several generations are born in a step
    mp.set_launch(**dict(mp.get_launch(), tail_passes=6))
    return dict(c=c, mp=mp)


def _ensemble(c, seed):
    """particles as a run holds them: swarm after swarm, some slots vacant, a few moved by
    compaction"""
    n, ns = c["n"], c["nswarm"]
    rng = np.random.default_rng(seed)
    a = np.zeros(n, dtype=STATE_DTYPE)
    a["x"] = rng.normal(scale=[0.02, 0.02, 0.05], size=(n, 3))
    T = np.exp(rng.uniform(math.log(1e4), math.log(1e7), n)) * co.eV
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    a["p"] = d * (np.sqrt((T + co.electron_mc2) ** 2 - co.electron_mc2 ** 2) / co.c)[:, None]
    a["w"] = rng.uniform(0.5, 2.0, n)
    a["uid"] = np.arange(n)
    sw = (np.arange(n, dtype=np.int64) * ns) // n
    moved = rng.random(n) < 0.02
    sw[moved] = rng.integers(0, ns, int(moved.sum()))
    a["swarm"] = sw
    a["active"] = rng.random(n) >= 0.05
    return a


def _prepare_statistics(c, seed):
    te, tg, tp = _air(dict(c, elo=0.4e6, ehi=4e6))
    mp = P.MultiPopulation(seed=seed, nswarm=c["nswarm"], electron=P.Population(c["n"], [], te, CUT),
                           photon=P.Population(1024, [], tg, CUT, tracked=False),
                           positron=P.Population(1024, [], tp, CUT, tracked=False))
    mp.set_particles(P.PT_ELECTRON, _ensemble(c, seed))
    return dict(c=c, mp=mp)


def prepare(case, seed):
    case = dict(case)
    return {"population": _prepare_population, "beam": _prepare_beam, "statistics": _prepare_statistics}[
        case["family"]](case, int(seed))


def _stats(mp, sp):
    s = mp.stats(sp)
    return {"count": np.array([s.n, s.nactive], dtype=np.int64),
            "moments": np.array([s.weight, s.mean_energy, s.max_energy, s.spread]), "centroid": np.array(s.centroid[:])}


def _state(mp, sp, rows):
    """the whole population in uid order, in arrays of a fixed number of rows (zeros after
    the last particle), as they are written to a file of a fixed layout"""
    a = mp.download(sp)
    a = a[np.argsort(a["uid"], kind="stable")]
    out = {}
    for f in ("x", "p", "w", "t", "s", "r", "uid"):
        out[f] = np.zeros((rows,) + a[f].shape[1:], dtype=a[f].dtype)
        out[f][: a.size] = a[f]
    return out


def _work(mp):
    w = mp.work(reset=True)
    return np.array([w.particle_steps, w.events, w.secondaries], dtype=np.int64)


class _Output(P.AbstractCallback):
    """what a run! script records at its outputs"""

    def __init__(self):
        self.rows = []

    def onoutput(self, mpopl, t=None, i=None):
        s = mpopl.stats(P.PT_ELECTRON)
        self.rows.append([t, float(s.nactive), s.weight, s.mean_energy])


def _run_population(s):
    c, mp = s["c"], s["mp"]
    mp.step = 0
    for sp in s["species"]:
        mp.set_particles(sp, EMPTY)
    uid = 0
    for i, k in enumerate(s["counts"]):
        mp.init_particles(P.PT_ELECTRON, k, c["e1"] * co.eV, (c["e2"] or c["e1"]) * co.eV, loguniform=c["e2"] > 0,
                          swarm=i, uid0=uid)
        uid += k
    mp.init()
    out = {}
    if c["mode"] == "loop":
        rec = _Output()
        cbs = [rec, P.PopulationTargetCallback("electron", 100 * c["n"])]
        if c["roulette"]:
            cbs.append(P.RouletteCallback(c["roulette"]))
        P.run_(mp, s["pusher"], (c["steps"] - 0.5) * DT, DT, P.CombinedCallback(cbs), output_dt=8 * DT, verbosity=0,
               compact_every=c["compact"])
        out["outputs"] = np.array(rec.rows)
    elif c["mode"] == "graph":
        mp.run_graph(0.0, DT, c["steps"], check_every=c["steps"])
    else:
        mp.run_steps(0.0, DT, c["steps"], compact_every=c["compact"], check_every=c["steps"])
    out["work"] = _work(mp)
    for sp in s["species"]:
        out["collisions%d" % sp] = mp.collision_counts(sp, reset=True)
        if c["state"]:
            out["state%d" % sp] = _state(mp, sp, c["n"] + c["n"] // 2 + 1024 if sp == 0 else c["n"] // 2 + 1024)
        else:
            out["stats%d" % sp] = _stats(mp, sp)
    if c["nswarm"] > 1:
        out["swarms"] = mp.swarm_stats(P.PT_ELECTRON)
    out["photon_births"] = mp.tally(P.PT_PHOTON)[0]
    return out


def _run_beam(s):
    c, mp = s["c"], s["mp"]
    mp.step = 0
    for sp in range(3):
        mp.set_particles(sp, EMPTY)
    mp.init_beam(P.PT_PHOTON, c["n"], 1e7 * co.eV)
    mp.init()
    mp.run_steps(0.0, 1e-9, c["steps"], compact_every=8, check_every=8)
    dose, under, over, total = mp.dose(reset=True)
    out = {"dose": dose, "dose_sums": np.array([under, over, total]), "photon_births": mp.tally(P.PT_PHOTON)[0],
           "work": _work(mp)}
    for sp in range(3):
        out["collisions%d" % sp] = mp.collision_counts(sp, reset=True)
        out["stats%d" % sp] = _stats(mp, sp)
    return out


def _run_statistics(s):
    mp = s["mp"]
    return {"stats": _stats(mp, P.PT_ELECTRON), "swarms": mp.swarm_stats(P.PT_ELECTRON)}


def run(state):
    return {"population": _run_population, "beam": _run_beam, "statistics": _run_statistics}[
        state["c"]["family"]](state)


def work(case):
    """What a pass cannot do without.  A particle's record is 93 bytes read and 72 written
    back; a push is about 150 double-precision operations and a collision (selection,
    sampling, rotation, next interval) about 400, 1.75 collisions per step of 1 ps.  A beam
    photon only flies; an electron in 1 ns has about 10^3 collisions."""
    n = case["n"]
    if case["family"] == "statistics":
        return {"bytes": n * (7 * 8 + 1 + 4), "flops": n * 30}
    if case["family"] == "beam":
        electrons = 0.0025 * n * case["steps"] ** 2  # summed over the steps
        return {"bytes": n * 165, "flops": n * case["steps"] * 150 + electrons * 1e3 * 400}
    return {"bytes": n * 165, "flops": n * case["steps"] * (150 + 1.75 * 400)}


def exact(case, seed):
    """64-bit values where there are such: the statistics of known particles.  A Monte Carlo
    run has none outside its own streams."""
    if case["family"] != "statistics":
        return None
    c = dict(case)
    a = _ensemble(c, int(seed))
    act = a["active"]
    b = a[act]
    L = np.longdouble
    light, mc2 = L(299792458.0), L(9.10938356e-31) * L(299792458.0) ** 2
    w, x, p = b["w"].astype(L), b["x"].astype(L), b["p"].astype(L)
    pc2 = (p * p).sum(1) * light ** 2
    E = pc2 / (np.sqrt(mc2 * mc2 + pc2) + mc2)
    W = w.sum()
    cen = (w[:, None] * x).sum(0) / W
    spread = np.sqrt(abs((w * (x * x).sum(1)).sum() / W - (cen * cen).sum()))
    sw = np.zeros((c["nswarm"], 4), dtype=np.float64)
    for i in range(c["nswarm"]):
        m = b["swarm"] == i
        if m.any():
            sw[i] = [m.sum(), w[m].sum(), (w[m] * E[m]).sum(), E[m].max()]
    return {"stats": {"count": np.array([a.size, int(act.sum())], dtype=np.int64),
                      "moments": np.array([W, (w * E).sum() / W, E.max(), spread]).astype(np.float64),
                      "centroid": cen.astype(np.float64)}, "swarms": sw}
