"""Device memory of a context: its slots, and the copy that a window of pt_run with late
compaction keeps."""
import ctypes as C

import numpy as np
import pytest
import torch

import helpers as H
import particulator_hip as P
from particulator_hip import co
from particulator_hip._lib import check, lib

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def device(caps):
    te, tg, tp = H.tables()
    return H.make_device(te, tg, tp, 5, caps=caps)


def test_slots_take_what_their_columns_take():
    """106 bytes a slot: a record of 80, uid, swarm, time left (where compaction also lists its
    positions), stream position and two flags.  All else (chunk counts, tables, counters, the
    launch's image, the allocator's rounding) is under 32 MiB."""
    caps = (1 << 24, (1 << 24) - 12345, 1 << 23)
    device((4096, 4096, 4096)).close()  # what the first context of a process sets up
    before = free()
    mp = device(caps)
    took = before - free()
    mp.close()
    assert took <= 106 * sum(caps) + 32 * MIB


def windows_of_each_species(n, room):
    """memory that three windows with late compaction take, each of another species"""
    mp = device((room, room, room))
    mp.init_particles(0, 1000, 2e6 * co.eV)
    mp.init()
    mp.run_steps(0.0, 1e-13, 3, compact_every=0, check_every=3)  # kernels loaded, no copy yet
    empty = np.zeros(0, dtype=P.population.STATE_DTYPE)
    before = free()
    for sp in range(3):
        for s in range(3):
            mp.set_particles(s, empty)
        mp.step = 0
        mp.init_particles(sp, n, 2e6 * co.eV)
        mp.init()
        mp.run_steps(0.0, 1e-14, 4, compact_every=1, check_every=4)
    took = before - free()
    out = (C.c_int64 * 4)()
    check(mp.ctx, lib().pt_debug_choices(mp.ctx, out))
    mp.close()
    assert out[2] == 3
    return took


def test_the_copy_of_late_compaction_is_bounded():
    """At most 2^21 particles of 93 bytes are copied aside, 186 MiB, whichever species they are
    of and in whatever order windows come.  (The first of two contexts takes what the runtime
    sets up once.)"""
    took = [windows_of_each_species(2_000_000, 4_100_000) for _ in range(2)][1]
    assert took <= 93 * (1 << 21) + 16 * MIB


def test_the_copy_is_given_back_when_memory_is_short():
    """An allocation that does not fit is tried again without the copy that an earlier window
    left (here it does not fit either: wall records beyond any GPU's memory), and the windows
    after it make a new one."""
    n, room = 1_500_000, 4_000_000
    mp = device((room, 4096, 4096))
    mp.init_particles(0, n, 2e6 * co.eV)
    mp.init()
    mp.run_steps(0.0, 1e-14, 4, compact_every=1, check_every=4)
    held = free()
    with pytest.raises(P.PTError) as e:
        mp.set_wall(0, 2, 1.0, capacity=1 << 38)
    assert e.value.code == -6
    assert free() - held >= 93 * n
    mp.run_steps(4e-14, 1e-14, 4, compact_every=1, check_every=4)
    assert free() - held <= 16 * MIB
    assert mp.stats(0).nactive > 0.9 * n
    mp.close()
