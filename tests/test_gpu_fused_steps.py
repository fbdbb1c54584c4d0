"""Several steps in one launch (pt_run, pt_run_graph) against one launch per step
(pt_advance): every random stream is keyed by (seed, uid, step) and a particle's steps
follow one another in registers exactly as they do through memory, so the populations
(matched by uid), the collision counters and the work counters must be equal, bit for bit.

The forms are those a launch tells apart: the field's reading (uniform in LDS, one swarm's
functor, several swarms' functors), continuum loss, restrictions, walls, long steps without
a force (the repeated pushes below the cut), populations below and across a wave, particles
that enter the run at different times, secondaries of several generations that overflow a
wave's stack, and step counts across the launch's limit."""
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


def pushers(form):
    if form == "swarms":
        return [P.RK2Pusher(EM(HF((0.0, 0.0, -e)))) for e in (4e5, 1e6, 4e6)]
    if form == "swarms of functors":
        return [P.RK2Pusher(EM(P.StepField(z, E0, (1e5, 0.0, 3e5)))) for z in (0.0, 1e-4)]
    if form == "layer and loss":
        return [P.RK2Pusher(P.CombinedForcing(EM(P.DoubleLayerField(-1e-3, 1e-3, E0), HF((0.0, 1e-2, 0.0))),
                                              air_loss(air.composition(), H.CUT, n=5)))]
    if form == "pushed photons only":
        return [P.RestrictedPusher("photon", P.RK2Pusher(EM(HF(E0))))]
    if form == "no force":
        return [P.RK2Pusher(EM(HF((0.0, 0.0, 0.0))))]
    return [P.RK2Pusher(EM(HF(E0)))]


#           form                   n   steps  dt     cut    energies       wall
FORMS = [("uniform", 1, 20, 1e-12, 1e4, (1e6, 1e6), None),
         ("uniform", 63, 9, 1e-12, 1e4, (1e5, 1e7), None),
         ("uniform", 5001, 37, 1e-12, 1e4, (1.2e4, 1e7), None),
         ("uniform", 4099, 12, 1e-12, 1e4, (1e5, 1e7), (2, 3e-4)),
         ("swarms", 3000, 17, 1e-12, 1e4, (1.5e4, 1e7), None),
         ("swarms of functors", 2050, 8, 1e-12, 1e4, (1e5, 1e7), None),
         ("layer and loss", 2050, 16, 1e-12, 1e4, (1.2e4, 1e7), None),
         ("pushed photons only", 1025, 8, 1e-12, 1e4, (1e5, 1e7), None),
         ("no force", 700, 5, 1e-9, 1e4, (1.2e4, 5e6), None),
         ("uniform", 1500, 4, 1e-10, 600.0, (1e5, 3e6), None)]


def run(form, n, steps, dt, cut_ev, energies, wall, mode):
    cut = cut_ev * co.eV
    ps = pushers(form)
    ns = len(ps)
    comp = air.composition()
    tabs = H.tables(dt=dt, cut=cut) if ns == 1 else air.swarm_tables(comp, [1e6] * ns, dt, cut)
    mp = H.make_device(*tabs, 77, caps=(1 << 20, 1 << 17, 1 << 16), cut=cut, nswarm=ns)
    for i, p in enumerate(ps):
        mp.set_pusher(p, swarm=i)
    for sp in range(3):
        m = max(1, n if sp == 0 else n // 8)
        init = O.init_swarm(m, sp, 5 + sp, uid0=sp * n, e1=energies[0], e2=energies[1], loguniform=True)
        soa, uid, _ = H.soa_of(init)
        soa[7, ::3] = 2.5 * dt  # every third particle enters in the third step
        mp.add_soa(sp, soa, uid=uid, swarm=np.arange(m) % ns)
    mp.init()
    if wall:
        mp.set_wall(0, wall[0], wall[1], drop=True, capacity=1 << 14)
    mp.work(reset=True)
    if mode == "steps":
        t = 0.0
        for _ in range(steps):
            mp.advance(t + dt)
            t += dt
    elif mode == "run":
        mp.run_steps(0.0, dt, steps, compact_every=0, check_every=steps)
    else:
        mp.set_launch(**dict(mp.get_launch(), compact_every=max(1, steps // 2)))
        mp.run_graph(0.0, dt, steps, check_every=steps)
    w = mp.work()
    out = dict(work=(w.particle_steps, w.events, w.secondaries, w.tail_particles), step=mp.step,
               counts=[mp.collision_counts(sp) for sp in range(3)], pop=[H.by_uid(mp.download(sp)) for sp in range(3)])
    if wall:
        out["wall"] = H.by_uid(mp.wall_records()[0])
    mp.close()
    return out


@pytest.mark.parametrize("form,n,steps,dt,cut,energies,wall", FORMS)
@pytest.mark.parametrize("mode", ["run", "graph"])
def test_steps_of_one_launch_equal_single_steps(form, n, steps, dt, cut, energies, wall, mode):
    a = run(form, n, steps, dt, cut, energies, wall, "steps")
    b = run(form, n, steps, dt, cut, energies, wall, mode)
    assert a["work"] == b["work"]
    assert a["step"] == b["step"] == steps
    for sp in range(3):
        assert np.array_equal(a["counts"][sp], b["counts"][sp])
        x, y = a["pop"][sp], b["pop"][sp]
        assert np.array_equal(x["uid"], y["uid"])
        for f in ("x", "p", "w", "t", "s", "r", "swarm"):
            assert np.array_equal(x[f], y[f]), (sp, f)
    if wall:
        x, y = a["wall"], b["wall"]
        assert x.size > 0 and np.array_equal(x["uid"], y["uid"])
        for f in ("x", "p", "t"):
            assert np.array_equal(x[f], y[f]), f


def test_single_steps_match_the_oracle_without_a_force():
    """The repeated pushes below the cut (no force, long steps) against the oracle, which
    does each of them: the particles dropped at the end of the step leave their energy
    where they stand, so the depth dose shows every push."""
    n, dt, seed = 400, 1e-9, 9
    te, tg, tp = H.tables(efield=0.0, dt=dt)
    init = O.init_swarm(n, 0, seed, e1=1.2e4, e2=3e4, loguniform=True)
    ow = H.make_oracle(te, tg, tp, seed, efield=(0.0, 0.0, 0.0))
    mp = H.make_device(te, tg, tp, seed, efield=(0.0, 0.0, 0.0))
    ow.add(0, init)
    ow.init()
    soa, uid, sw = H.soa_of(init)
    mp.add_soa(0, soa, uid=uid, swarm=sw)
    mp.init()
    ow.advance(dt)
    mp.advance(dt)
    a, b = H.by_uid(ow.particles(0)), H.by_uid(mp.download(0))
    assert abs(a.size - b.size) <= 2
    dropped = H.by_uid(mp.download(0, active_only=False))
    # every electron of this energy loses most of it in 1 ns, and each ends its step at dt
    assert dropped.size > b.size
    assert np.all(np.abs(dropped["t"] - dt) <= 4.5e-16)
