"""The wide workgroups of large populations against the small ones (a launch of block 128
never uses them): random streams are keyed by (seed, uid, step), so populations (matched by
uid), collision counters and work counters must be equal, bit for bit, and the depth dose up
to the order of its sums.

Sizes lie on both sides of the rule (four electrons and positrons per lane of a launch of 256
CUs, 786,432; 1.5 in launches of one step) and are ragged; the forms are those whose values the wide kernel reads from LDS
or memory instead of registers: one swarm's force, several swarms' forces and rate bounds, a
magnetic field, functors, continuum loss, and electrons with positrons and photons."""
import numpy as np
import pytest

import helpers as H
import oracle as O
import particulator_hip as P
from particulator_hip import air, co
from particulator_hip.continuum import air_loss

pytestmark = pytest.mark.gpu

HF = P.HomogeneousField
EM = P.ElectromagneticField
E0 = (0.0, 0.0, -1e6)
LINE = 4 * 768 * 256


def pushers(form):
    if form == "swarms":
        return [P.RK2Pusher(EM(HF((0.0, 0.0, -e)))) for e in (4e5, 1e6, 4e6)]
    if form == "swarms, E across":
        return [P.RK2Pusher(EM(HF((3e5, -1e5, -e)))) for e in (4e5, 1e6, 4e6)]
    if form == "swarms with B":
        return [P.RK2Pusher(EM(HF((0.0, 0.0, -e)), HF((0.0, 1e-2, 0.0)))) for e in (4e5, 1e6)]
    if form == "swarms of functors":
        return [P.RK2Pusher(EM(P.StepField(z, E0, (1e5, 0.0, 3e5)))) for z in (0.0, 1e-4)]
    if form == "layer and loss":
        return [P.RK2Pusher(P.CombinedForcing(EM(P.DoubleLayerField(-1e-3, 1e-3, E0), HF((0.0, 1e-2, 0.0))),
                                              air_loss(air.composition(), H.CUT, n=5)))]
    if form == "no force on electrons":
        return [P.RestrictedPusher("positron", P.RK2Pusher(EM(HF(E0))))]
    return [P.RK2Pusher(EM(HF(E0)))]


def run(form, n, steps, mode, block, seed=31, dt=1e-12):
    ps = pushers(form)
    ns = len(ps)
    comp = air.composition()
    tabs = H.tables(dt=dt) if ns == 1 else air.swarm_tables(comp, [1e6] * ns, dt, H.CUT)
    pops = {name: P.Population(cap, [], tb, H.CUT, tracked=True)
            for name, tb, cap in zip(("electron", "photon", "positron"), tabs, (1 << 21, 1 << 19, 1 << 18))}
    mp = P.MultiPopulation(seed=seed, nswarm=ns, dose=(64, -1e-3, 1e-3), **pops)
    for i, p in enumerate(ps):
        mp.set_pusher(p, swarm=i)
    uid0 = 0
    for sp, m in ((0, n - n // 10), (1, n // 16), (2, n // 10)):
        soa, uid, _ = H.soa_of(O.init_swarm(m, sp, 5 + sp, uid0=uid0, e1=1.2e4, e2=1e7, loguniform=True))
        mp.add_soa(sp, soa, uid=uid, swarm=np.arange(m) % ns)
        uid0 += m
    mp.init()
    mp.set_launch(**dict(mp.get_launch(), block=block, compact_every=4))
    mp.work(reset=True)
    if mode == "steps":
        for k in range(steps):
            mp.advance((k + 1) * dt)
    elif mode == "run":
        mp.run_steps(0.0, dt, steps, compact_every=3, check_every=steps)
    else:
        mp.run_graph(0.0, dt, steps, check_every=steps)
    w = mp.work()
    out = dict(work=(w.particle_steps, w.events, w.secondaries), dose=mp.dose(),
               counts=[mp.collision_counts(sp) for sp in range(3)], pop=[H.by_uid(mp.download(sp)) for sp in range(3)])
    mp.close()
    return out


@pytest.mark.parametrize("form,n,steps,mode", [
    ("uniform", LINE * 3 // 8 - 1, 3, "steps"), ("uniform", LINE * 3 // 8, 3, "steps"),
    ("uniform", LINE - 1, 3, "run"), ("uniform", LINE, 3, "run"), ("uniform", LINE + 12345, 8, "run"),
    ("uniform", LINE + 1, 9, "graph"), ("swarms", LINE + 77, 5, "run"), ("swarms, E across", LINE + 63, 3, "run"),
    ("swarms with B", LINE + 65, 3, "run"), ("swarms of functors", LINE + 7, 2, "run"),
    ("layer and loss", LINE + 129, 3, "graph"), ("no force on electrons", LINE + 5, 5, "run")])
def test_wide_workgroups_equal_small_ones(form, n, steps, mode):
    a = run(form, n, steps, mode, 128)
    b = run(form, n, steps, mode, 256)
    assert a["work"] == b["work"] and a["work"][1] > 0
    for sp in range(3):
        assert np.array_equal(a["counts"][sp], b["counts"][sp])
        x, y = a["pop"][sp], b["pop"][sp]
        assert x.size > 0 and np.array_equal(x["uid"], y["uid"])
        for f in ("x", "p", "w", "t", "s", "r", "swarm"):
            assert np.array_equal(x[f], y[f]), (sp, f)
    # the bins are sums of at most a few 10^5 positive terms in any order (n eps/2 each way)
    assert np.allclose(a["dose"][0], b["dose"][0], rtol=1e-10, atol=0.0)
    assert np.allclose(a["dose"][1:], b["dose"][1:], rtol=1e-9, atol=0.0)


@pytest.mark.parametrize("n", [256 * 256 - 1, 256 * 256, 256 * 256 + 1])
@pytest.mark.parametrize("block", [128, 256, 512])
def test_one_wave_per_simd_equals_the_full_launch(n, block):
    """Particles of all species up to one per lane of a single wave per SIMD (65,536): the
    launches of pt_run against those of a captured run, which always fill the GPU."""
    m = n - n // 17  # (run() adds n // 16 photons)
    a = run("uniform", m, 6, "run", block)
    b = run("uniform", m, 6, "graph", block)
    assert a["work"] == b["work"] and a["work"][1] > 0
    for sp in range(3):
        assert np.array_equal(a["counts"][sp], b["counts"][sp])
        x, y = a["pop"][sp], b["pop"][sp]
        assert np.array_equal(x["uid"], y["uid"])
        for f in ("x", "p", "w", "t", "s", "r", "swarm"):
            assert np.array_equal(x[f], y[f]), (sp, f)


@pytest.mark.parametrize("photons", [4 * 65536 - 1, 4 * 65536, 300_001])
def test_a_beam_on_one_wave_per_simd_equals_the_full_launch(photons):
    """Photons with few electrons run on one wave per SIMD from four per lane on; a launch of
    two workgroups per resident one (grid_mult 2) never does."""
    out = []
    for mult in (1, 2):
        te, tg, tp = H.tables()
        mp = H.make_device(te, tg, tp, 3, caps=(1 << 17, 1 << 19, 1 << 15))
        soa, uid, _ = H.soa_of(O.init_swarm(photons, 1, 7, e1=2e4, e2=5e6, loguniform=True))
        mp.add_soa(1, soa, uid=uid, swarm=np.zeros(photons, np.int32))
        mp.init()
        mp.set_launch(**dict(mp.get_launch(), grid_mult=mult))
        mp.run_steps(0.0, 2e-11, 6, compact_every=3, check_every=6)
        out.append([H.by_uid(mp.download(sp)) for sp in range(3)] + [mp.collision_counts(sp) for sp in range(3)])
        mp.close()
    a, b = out
    assert a[0].size > 0 and a[1].size < photons
    for sp in range(3):
        assert np.array_equal(a[3 + sp], b[3 + sp])
        assert np.array_equal(a[sp]["uid"], b[sp]["uid"])
        for f in ("x", "p", "w", "t", "s", "r", "swarm"):
            assert np.array_equal(a[sp][f], b[sp][f]), (sp, f)
