"""The largest tables that pt_upload_table takes (24 processes, 62 and 63 intervals, three species) with
several swarms and a depth dose: the step's workgroups of every size the caller may ask for,
captured runs, collision rounds and the last passes over secondaries have to find room for
them in LDS.  The particles do not depend on the launch, so every way has to end as single
steps of 128-thread workgroups do."""
import numpy as np
import pytest

import helpers as H
import oracle as O
import particulator_hip as P
from particulator_hip import air, co
from particulator_hip.physics import RelativisticCoulomb
from particulator_hip.tables import collision_table_from_processes

pytestmark = pytest.mark.gpu

DT = 1e-12
NPROCS = 24


def tables(nswarm, intervals):
    comp = air.composition()
    F = co.elementary_charge * 1e6 * DT
    out = []
    for sp, procs, f in ((0, air.electron_processes(comp, H.CUT), F), (1, air.photon_processes(comp), 0.0),
                         (2, air.positron_processes(comp, H.CUT), F)):
        procs = list(procs)
        # the table filled up with rarer scatterers of the kinds that are there
        extra = procs if sp == 1 else [(c, p) for c, p in procs if isinstance(p, RelativisticCoulomb)]
        while len(procs) < NPROCS:
            c, p = extra[len(procs) % len(extra)]
            procs.append((1e-3 * c, p))
        with np.errstate(all="ignore"):
            t = collision_table_from_processes(procs, sp, f, nintervals=intervals, energy_cut=H.CUT)
        # (of the lowest intervals, far below the cut, nothing is used)
        for a in (t.rate, t.ratebound):
            a[~np.isfinite(a)] = 0.0
        out.append(t.with_ratebounds(np.repeat(t.ratebound, nswarm, axis=0)) if sp != 1 and nswarm > 1 else t)
    return out


def run(tabs, nswarm, dose, mode, homogeneous, **launch):
    caps = (1 << 14, 1 << 13, 1 << 12)
    pops = {n: P.Population(c, [], t, H.CUT, tracked=True)
            for n, t, c in zip(("electron", "photon", "positron"), tabs, caps)}
    mp = P.MultiPopulation(seed=12, nswarm=nswarm, dose=(dose, -1e-3, 1e-3) if dose else None, **pops)
    for i in range(nswarm):
        e = P.HomogeneousField((0.0, 1e4 * i, -1e6))
        b = P.HomogeneousField((0.0, 1e-3, 0.0))
        step = P.StepField(1e-4 * i, (0.0, 0.0, -1e6), (1e5, 0.0, 3e5))
        f = P.ElectromagneticField(e, b) if homogeneous else P.ElectromagneticField(step)
        mp.set_pusher(P.RK2Pusher(f), swarm=i)
    uid0 = 0
    for sp, m in ((0, 1500), (1, 300), (2, 301)):
        soa, uid, _ = H.soa_of(O.init_swarm(m, sp, 5 + sp, uid0=uid0, e1=2e4, e2=1e7, loguniform=True))
        mp.add_soa(sp, soa, uid=uid, swarm=np.arange(m) % nswarm)
        uid0 += m
    mp.init()
    mp.set_launch(**dict(mp.get_launch(), compact_every=2, **launch))
    if mode == "steps":
        for k in range(5):
            mp.advance((k + 1) * DT)
    elif mode == "run":
        mp.run_steps(0.0, DT, 5, compact_every=2, check_every=5)
    else:
        mp.run_graph(0.0, DT, 5, check_every=5)
    out = [H.by_uid(mp.download(sp)) for sp in range(3)] + [mp.collision_counts(sp) for sp in range(3)]
    mp.close()
    return out


@pytest.mark.parametrize("nswarm,dose,homogeneous,intervals", [
    (1, 0, True, 63), (1, 0, True, 32), (2, 0, False, 61), (2, 0, False, 62), (2, 0, False, 63), (2, 512, False, 60),
    (2, 512, False, 63), (256, 512, True, 63)])
def test_every_launch_finds_room(nswarm, dose, homogeneous, intervals):
    tabs = tables(nswarm, intervals)
    assert all(len(t) == NPROCS and t.b.k == intervals for t in tabs)
    a = run(tabs, nswarm, dose, "steps", homogeneous, block=128)
    assert a[0].size > 1000 and a[3][1:].sum() > 1000
    for mode, launch in (("run", dict(block=128)), ("run", dict(block=256)), ("run", dict(block=512)),
                         ("steps", dict(block=512)), ("graph", dict(block=256)), ("graph", dict(block=512)),
                         ("run", dict(block=256, rounds=1)), ("run", dict(block=512, rounds=2))):
        b = run(tabs, nswarm, dose, mode, homogeneous, **launch)
        for sp in range(3):
            assert np.array_equal(a[3 + sp], b[3 + sp]), (mode, launch)
            assert np.array_equal(a[sp]["uid"], b[sp]["uid"]), (mode, launch)
            for f in ("x", "p", "w", "t"):
                assert np.array_equal(a[sp][f], b[sp][f]), (mode, launch, sp, f)
