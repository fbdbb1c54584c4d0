"""Compaction (repack!) at the edges of its chunks and of its 16-byte reads, for every pattern
of vacant slots, and a run whose compactions wait until the end of a launch: it must end as
the same run compacted step by step does, also when a population would not fit without the
slots that those compactions free."""
import numpy as np
import pytest

import helpers as H
import oracle as O
from particulator_hip import co
from particulator_hip._lib import PTError
from particulator_hip.population import STATE_DTYPE

pytestmark = pytest.mark.gpu


def population(n, pattern, rng):
    a = np.zeros(n, dtype=STATE_DTYPE)
    a["x"] = rng.normal(size=(n, 3))
    a["p"] = rng.normal(size=(n, 3)) * 1e-21
    a["w"], a["s"], a["t"] = rng.uniform(size=(3, n))
    a["uid"] = rng.permutation(n).astype(np.uint64) + np.uint64(1 << 40)
    i = np.arange(n)
    a["active"] = {"all": i >= 0, "none": i < 0, "one": i == n - 1, "first half": i < n // 2, "second half": i >= n // 2,
                   "odd": i % 2 == 1, "random": rng.random(n) < 0.3, "few vacant": rng.random(n) < 0.999}[pattern]
    return a


@pytest.mark.parametrize("n", [1, 15, 17, 4095, 4096, 4097, 12289, 300_001])
def test_compaction_keeps_the_actives(n):
    te, tg, tp = H.tables()
    rng = np.random.default_rng(n)
    mp = H.make_device(te, tg, tp, 1, caps=(n, n + 3, 2 * n))
    patterns = ["all", "none", "one", "first half", "second half", "odd", "random", "few vacant"]
    for k, pattern in enumerate(patterns):
        pops = [population(n, patterns[(k + s) % len(patterns)], rng) for s in range(3)]
        for s in range(3):
            mp.set_particles(s, pops[s])
        mp.compact(-1 if k % 2 else 0)
        for s in range(3):
            done = k % 2 or s == 0
            want = H.by_uid(pops[s][pops[s]["active"]])
            assert mp.count(s) == (want.size if done else n)
            got = H.by_uid(mp.download(s))
            for f in ("uid", "x", "p", "w", "t", "s", "r", "swarm"):
                assert np.array_equal(got[f], want[f]), (pattern, s, f)
    mp.close()


def device(seed, cap, n, dt, cut):
    te, tg, tp = H.tables(dt=dt, cut=cut)
    mp = H.make_device(te, tg, tp, seed, caps=(cap, 1 << 14, 1 << 12), cut=cut)
    init = O.init_swarm(n, 0, seed, e1=1.5e4, e2=4e4, loguniform=True)
    soa, uid, sw = H.soa_of(init)
    mp.add_soa(0, soa, uid=uid, swarm=sw)
    mp.init()
    return mp


def result(mp):
    w = mp.work()
    return dict(work=(w.particle_steps, w.events, w.secondaries), step=mp.step, counts=[mp.count(s) for s in range(3)],
                coll=[mp.collision_counts(s) for s in range(3)], pop=[H.by_uid(mp.download(s)) for s in range(3)])


@pytest.mark.parametrize("every,steps", [(1, 40), (3, 40), (5, 33)])
def test_late_compaction_ends_as_compaction_in_time(every, steps):
    """Electrons that live for a few steps and leave secondaries: the slots in use between
    compactions exceed the population's capacity unless each compaction comes in time."""
    seed, n, dt, cut = 19, 300, 3e-11, 600.0 * co.eV
    ref = device(seed, 1 << 16, n, dt, cut)
    t, need = 0.0, 0
    for q in range(steps):
        ref.advance(t + dt)
        t += dt
        need = max(need, ref.count(0))
        if (q + 1) % every == 0:
            ref.compact(-1)
    a = result(ref)
    ref.close()
    for cap in (max(need, 2 * n), 1 << 16):
        mp = device(seed, cap, n, dt, cut)
        mp.run_steps(0.0, dt, steps, compact_every=every, check_every=steps)
        b = result(mp)
        assert a["work"] == b["work"] and a["step"] == b["step"] and a["counts"] == b["counts"]
        for s in range(3):
            assert np.array_equal(a["coll"][s], b["coll"][s])
            for f in ("uid", "x", "p", "w", "t", "s", "r"):
                assert np.array_equal(a["pop"][s][f], b["pop"][s][f]), (s, f)
        mp.close()
    # the smaller capacity does not hold the particles of a whole run: without compactions
    # in time the run would have failed
    assert n + a["work"][2] > max(need, 2 * n)
    # and one that does not hold them in any case is still refused
    if need > 2 * n:
        mp = device(seed, need - 1, n, dt, cut)
        with pytest.raises(PTError):
            mp.run_steps(0.0, dt, steps, compact_every=every, check_every=steps)
        mp.close()
