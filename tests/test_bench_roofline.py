"""The bench line's roofline: a launch of several steps moves each particle once, so the bytes
it has to move do not grow with its steps."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import bench  # noqa: E402


def test_bytes_of_a_launch_do_not_grow_with_its_steps():
    n, per_step = 10_000_000, 3000
    for k in (1, 8, 16):
        steps = 48
        got = bench.launch_bytes(n * steps, per_step * steps, steps, steps // k)
        assert got == pytest.approx(165.0 * n + 93.0 * per_step * k, rel=1e-12)


def test_the_bound_is_instruction_issue():
    traffic = {"bytes": 1.96e9, "valu": {"wave_instructions_per_particle_step": 64.0, "simds": 1024}}
    r = bench.roofline(psteps=8e7, secondaries=0, steps=8, launches=1, avg_launch_ms=10.0, rate=8e9, traffic=traffic)
    assert r["peak"] == pytest.approx(614.4) and r["achieved"] == pytest.approx(512.0)
    assert r["frac"] == pytest.approx(512.0 / 614.4)
    assert r["hbm"]["achieved"] == pytest.approx(165.0)
    # without counters there is no figure for it
    r = bench.roofline(8e7, 0, 8, 1, 10.0, 8e9, None)
    assert r["achieved"] is None and r["frac"] is None and r["hbm"]["achieved"] == pytest.approx(165.0)
