"""Particles below the cut in long steps: one that a collision leaves there flies on freely, one
that the field decelerates there goes on in pushes of s / r until the step's end (s is not
drawn again, src/collisions.jl:151).  The end points of all slots, those of the dropped
particles among them, against the oracle and against collision rounds."""
import numpy as np
import pytest

import helpers as H
import oracle as O
import particulator_hip as P
from particulator_hip import co

pytestmark = pytest.mark.gpu

def device(n, seed, field, dt, e1, e2, dose=None, caps=(1 << 16, 1 << 14, 1 << 12), **launch):
    te, tg, tp = H.tables(efield=field, dt=dt)
    pops = {name: P.Population(cap, [], tb, H.CUT, tracked=True)
            for name, tb, cap in zip(("electron", "photon", "positron"), (te, tg, tp), caps)}
    mp = P.MultiPopulation(seed=seed, dose=dose, **pops)
    mp.set_pusher(P.RK2Pusher(P.ElectromagneticField(P.HomogeneousField((0.0, 0.0, -field)))))
    mp.set_launch(**dict(mp.get_launch(), **launch))
    init = O.init_swarm(n, 0, seed, e1=e1, e2=e2, loguniform=True)
    soa, uid, sw = H.soa_of(init)
    mp.add_soa(0, soa, uid=uid, swarm=sw)
    mp.init()
    return mp, init


#          V/m  step   energies    least share that ends below the cut
CASES = [(0.0, 1e-9, 1.2e4, 3e4, 0.9), (1e6, 1e-11, 1e4, 1.5e4, 0.2), (4e6, 1e-11, 1e4, 2e4, 0.1)]


@pytest.mark.parametrize("field,dt,e1,e2,share", CASES)
def test_end_points_match_the_oracle(field, dt, e1, e2, share):
    """One step of electrons that collide some tens of times and lose a few keV.  A collision's
    rounding is about 1e-15 of the momentum, so after up to 10^3 of them, each amplified by at
    most 10^2 through the next one's angles and rates, end points agree to 1e-10 of the path;
    1e-9 is asked of all but 1%, whose history a rounding may have turned at a selection."""
    n, seed = 400, 9
    mp, init = device(n, seed, field, dt, e1, e2)
    ow = H.make_oracle(*H.tables(efield=field, dt=dt), seed, efield=(0.0, 0.0, -field))
    ow.add(0, init)
    ow.init()
    ow.advance(dt, droplow=False)
    mp.advance(dt)
    a, b = H.by_uid(ow.particles(0, active_only=False)), H.by_uid(mp.download(0, active_only=False))
    both, ia, ib = np.intersect1d(a["uid"], b["uid"], return_indices=True)
    assert both.size >= 0.99 * max(a.size, b.size)
    a, b = a[ia], b[ib]
    path = 0.3 * co.c * dt  # at most the speed of 30 keV
    dx = np.abs(a["x"] - b["x"]).max(axis=1)
    dp = np.abs(a["p"] - b["p"]).max(axis=1) / np.abs(a["p"]).max(axis=1)
    good = (dx <= 1e-9 * path) & (dp <= 1e-9) & (np.abs(a["t"] - b["t"]) <= 1e-9 * dt)
    assert good.sum() >= 0.99 * both.size
    # many end below the cut, and away from where they began
    below = P.population.kinenergy(0, b["p"]) < H.CUT
    assert below.sum() > share * n and np.linalg.norm(b["x"], axis=1)[below].min() > 0.0
    assert np.all(~b["active"][below])
    mp.close()


@pytest.mark.parametrize("field,dt,e1", [c[:3] for c in CASES])
@pytest.mark.parametrize("steps", [1, 3])
def test_end_points_equal_those_of_collision_rounds(field, dt, e1, steps):
    """bit for bit, also over several steps of one launch; the dose up to the order of its sums"""
    out = []
    for launch in (dict(rounds=0), dict(rounds=1, defer_mask=(1 << 2) | (1 << 4))):
        mp, _ = device(700, 23, field, dt, e1, 5e6 if field == 0.0 else 2e4, dose=(64, -0.5, 0.5), **launch)
        mp.run_steps(0.0, dt, steps, compact_every=0, check_every=steps)
        out.append([H.by_uid(mp.download(sp, active_only=False)) for sp in range(3)] + [mp.dose()])
        mp.close()
    a, b = out
    for sp in range(3):
        assert np.array_equal(a[sp]["uid"], b[sp]["uid"])
        for f in ("x", "p", "w", "t", "active"):
            assert np.array_equal(a[sp][f], b[sp][f]), (sp, f)
    assert (~a[0]["active"]).sum() > 100
    # sums of some 10^5 positive terms in any order
    assert np.allclose(a[3][0], b[3][0], rtol=1e-10, atol=0.0)
    assert a[3][0].sum() > 0.0
