"""The paths that the library chooses by itself, as pt_debug_choices reports them: the shape of
the main pass's launch on both sides of its rules, and the windows of pt_run that compact
late or are taken back.  (That the results do not depend on them is tested in
test_gpu_wide.py and test_gpu_compaction.py.)"""
import ctypes as C

import numpy as np
import pytest
import torch

import helpers as H
import oracle as O
import particulator_hip as P
from particulator_hip import air, co
from particulator_hip._lib import check, lib

pytestmark = pytest.mark.gpu


def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def choices(mp):
    out = (C.c_int64 * 4)()
    check(mp.ctx, lib().pt_debug_choices(mp.ctx, out))
    return dict(block=out[0], waves=out[0] // 64 * out[1], late=out[2], back=out[3])


def electrons(n, block, dt=1e-12, grid_mult=1):
    te, tg, tp = H.tables()
    mp = H.make_device(te, tg, tp, 3, caps=(2 * n + 4096, n // 2 + 4096, 4096))
    mp.init_particles(0, n, 1e5 * co.eV, 1e6 * co.eV, loguniform=True)
    mp.init()
    mp.set_launch(**dict(mp.get_launch(), block=block, grid_mult=grid_mult))
    return mp


@pytest.mark.parametrize("mode,eighths", [("run", 32), ("graph", 32), ("advance", 12)])
@pytest.mark.parametrize("block", [128, 256, 512])
def test_large_populations_run_in_wide_workgroups(mode, eighths, block):
    """Four electrons per lane of a 768-thread workgroup on each CU, 1.5 for one step alone; a
    caller's workgroups of 128 threads stay as they are."""
    line = eighths * 768 * cus() // 8
    for n, wide in ((line - 1, False), (line, block != 128)):
        mp = electrons(n, block)
        if mode == "advance":
            mp.advance(1e-12)
        elif mode == "run":
            mp.run_steps(0.0, 1e-12, 2, check_every=2)
        else:
            mp.run_graph(0.0, 1e-12, 8, check_every=8)
        c = choices(mp)
        assert c["block"] == (768 if wide else block), n
        mp.close()


@pytest.mark.parametrize("block", [128, 256, 512])
def test_small_populations_run_on_one_wave_per_simd(block):
    """A particle per lane of four waves on each CU or fewer; not beyond, not in captured runs,
    and not in workgroups of 512 threads, eight waves each.  (The wide rule lies far above.)"""
    line = 256 * cus()
    for n in (1000, line, line + 1):
        mp = electrons(n, block)
        mp.run_steps(0.0, 1e-12, 2, check_every=2)
        one = choices(mp)["waves"]
        assert (one <= 4 * cus()) == (n <= line and block != 512), n
        mp.run_graph(0.0, 1e-12, 8, check_every=8)
        assert choices(mp)["waves"] > 4 * cus()
        mp.close()


@pytest.mark.parametrize("mode", ["run", "advance"])
@pytest.mark.parametrize("per_lane,more,dt,thin,one", [
    (4, -1, 1e-9, 1.0, False), (4, 0, 1e-12, 1.0, True), (16, 0, 1e-12, 1.0, True), (16, 1, 1e-12, 1.0, False),
    (16, 1, 1e-10, 1.0, False), (16, 1, 1e-9, 1.0, True), (16, 1, 1e-9, 1e-2, False), (128, 0, 1e-9, 1.0, True),
    (128, 1, 1e-9, 1.0, False)])
def test_beams_run_on_one_wave_per_simd(mode, per_lane, more, dt, thin, one):
    """Photons and no electrons: from 4 per lane to 16 whatever the step, to 128 with long steps
    in dense air"""
    n = per_lane * 256 * cus() + more
    comp = {k: v * thin for k, v in air.composition().items()}
    te, tg, tp = H.tables(efield=0.0, dt=dt, comp=comp)
    mp = H.make_device(te, tg, tp, 3, caps=(1 << 18, n + n // 16, 1 << 16))
    mp.init_beam(1, n, 1e5 * co.eV)
    mp.init()
    if mode == "advance":
        mp.advance(dt)
    else:
        mp.run_steps(0.0, dt, 2, check_every=2)
    assert (choices(mp)["waves"] <= 4 * cus()) == one
    mp.close()


def test_autotuner_keeps_the_smaller_of_equal_launches():
    """A large population runs the same wide workgroups for 256 and 512: the trials of 512 are
    repetitions, and none of their rates, differing by noise, is chosen."""
    mp = electrons(4 * 768 * cus() + 100_000, 256)
    best, trials, _ = mp.autotune(0.0, 1e-13, trial_steps=2)
    assert [t["block"] for t in trials[4:13]] == [128] * 3 + [256] * 3 + [512] * 3
    assert best["block"] != 512 or best["rounds"] > 0
    mp.close()


def late(cap, n, dt, every, steps):
    cut = 600.0 * co.eV
    te, tg, tp = H.tables(dt=dt, cut=cut)
    mp = H.make_device(te, tg, tp, 19, caps=(cap, 1 << 14, 1 << 12), cut=cut)
    soa, uid, sw = H.soa_of(O.init_swarm(n, 0, 19, e1=1.5e4, e2=4e4, loguniform=True))
    mp.add_soa(0, soa, uid=uid, swarm=sw)
    mp.init()
    return mp


@pytest.mark.parametrize("every,steps", [(1, 40), (3, 40), (5, 33)])
def test_windows_compact_late_and_are_taken_back(every, steps):
    """Electrons that live for a few steps and leave secondaries.  The smallest capacity that
    the compactions asked for allow holds no launch of 16 steps without them: its window is
    taken back.  A capacity that holds the whole run's particles takes none back."""
    n, dt = 300, 3e-11
    ref = late(1 << 16, n, dt, every, steps)
    t, need, most, base, first = 0.0, 0, 0, n, 0
    for q in range(steps):
        ref.advance(t + dt)
        t += dt
        need = max(need, ref.count(0))
        # the slots a launch over the steps since its start would need (late compaction comes
        # after 16 steps, or at the window's last compaction)
        w = ref.work()
        most = max(most, base + w.secondaries - first)
        if (q + 1) % every == 0:
            ref.compact(-1)
        if (q + 1) % 16 == 0:
            base, first = int(ref.stats(0).nactive), w.secondaries
    ref.close()
    tight = max(need, 2 * n)
    assert most > tight  # (electrons are nearly all of the secondaries)
    for cap, back in ((tight, 1), (1 << 16, 0)):
        mp = late(cap, n, dt, every, steps)
        mp.run_steps(0.0, dt, steps, compact_every=every, check_every=steps)
        c = choices(mp)
        assert (c["late"], c["back"]) == (1, back), cap
        mp.close()


def test_windows_that_never_compact_late():
    n, dt = 300, 3e-11
    for every, steps, cap in ((0, 20, 1 << 16), (16, 40, 1 << 16), (1, 1, 1 << 16), (1, 20, 2 * n - 1)):
        mp = late(cap, n, dt, every, 1)
        try:
            mp.run_steps(0.0, dt, steps, compact_every=every, check_every=steps)
        except P.PTError:
            assert cap < 2 * n
        assert choices(mp)["late"] == 0
        mp.close()


def test_choices_refuses_null():
    mp = late(1 << 12, 1, 1e-12, 1, 1)
    assert lib().pt_debug_choices(None, (C.c_int64 * 4)()) == -1
    assert lib().pt_debug_choices(mp.ctx, None) == -1
    mp.close()
