"""Per-swarm sums of populations on both sides of the size from which the workgroups add into
several arrays (128 workgroups of 256), called repeatedly and with fewer swarms in between:
the arrays are cleared by the call that used them."""
import numpy as np
import pytest

import helpers as H
from particulator_hip import co
from particulator_hip.population import STATE_DTYPE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 127 * 256, 127 * 256 + 1, 128 * 256, 200_003])
@pytest.mark.parametrize("ns", [1, 5, 1024, 1025])
def test_swarm_sums(n, ns):
    te, tg, tp = H.tables()
    rng = np.random.default_rng(n + ns)
    a = np.zeros(n, dtype=STATE_DTYPE)
    a["p"] = rng.normal(size=(n, 3)) * 1e-22
    a["w"] = rng.uniform(0.5, 2.0, n)
    a["uid"] = np.arange(n)
    a["swarm"] = (np.arange(n, dtype=np.int64) * ns) // n
    moved = rng.random(n) < 0.02
    a["swarm"][moved] = rng.integers(0, ns, int(moved.sum()))
    a["active"] = rng.random(n) >= 0.05
    mp = H.make_device(te, tg, tp, 5, caps=(max(n, 64), 64, 64), nswarm=ns)
    mp.set_particles(0, a)
    m = a["active"] != 0
    E = np.sqrt((a["p"] ** 2).sum(axis=1) * co.c ** 2 + co.electron_mc2 ** 2) - co.electron_mc2
    want = np.zeros((ns, 4))
    for q, v in enumerate((np.ones(n), a["w"], a["w"] * E)):
        want[:, q] = np.bincount(a["swarm"][m], weights=v[m], minlength=ns)
    np.maximum.at(want[:, 3], a["swarm"][m], E[m])
    for k in (ns, max(1, ns // 2), ns, ns):
        got = mp.swarm_stats(0, k)
        assert np.array_equal(got[:, 0], want[:k, 0])
        # (an energy is a difference: its relative error is eps mc^2 / E, 1e-14 at 1e-22 kg m/s)
        assert np.allclose(got, want[:k], rtol=1e-10, atol=0.0)
    mp.close()
