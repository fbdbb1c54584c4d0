"""The selection scan over cumulative rates against the scan over rates it stands for
(src/collisions.jl:160-186), on tables of 1 to 24 processes: whole and ragged groups, rates
that are zero, negative or not a number in part of the table, null collisions, the first and
the last interval.

The two sums differ by rounding: an energy and draw whose decision lies within 1e-12 of the
total rate (2 x 24 additions of eps/2 = 5e-15, and as much again for the coefficients, with
room) is left out."""
import ctypes as C

import numpy as np
import pytest

import helpers as H
from particulator_hip import co
from particulator_hip._lib import check, lib
from particulator_hip.tables import ChebyshevCollisionTable

pytestmark = pytest.mark.gpu


def table(base, nproc, kind, seed):
    rng = np.random.default_rng(seed)
    k1 = base.b.k + 1
    rate = rng.uniform(0.2, 2.0, (k1, nproc, 3)) * 10.0 ** rng.uniform(-4, 0, (1, nproc, 1))
    rate[..., 1:] *= 0.2
    if kind == "zeros":
        rate[:, rng.random(nproc) < 0.4] = 0.0
    elif kind == "negative":
        rate[rng.random((k1, nproc)) < 0.3] *= -0.3
    elif kind == "NaN rows":
        rate[1::2] = np.nan
    rb = np.zeros((1, k1, 3))
    rb[0, :, 0] = 1.2 * np.nan_to_num(np.abs(rate)).sum(axis=(1, 2)).max() + 1e-3
    return ChebyshevCollisionTable([base.proc[q % len(base.proc)] for q in range(nproc)], base.b, rate, rb, base.species)


@pytest.mark.parametrize("nproc", [1, 2, 3, 4, 5, 6, 7, 23, 24])
@pytest.mark.parametrize("kind", ["plain", "zeros", "negative", "NaN rows"])
def test_selection_matches_the_sequential_scan(nproc, kind):
    te, tg, tp = H.tables()
    tb = table(te, nproc, kind, 100 + nproc)
    mp = H.make_device(tb, tg, tp, 5)
    rng = np.random.default_rng(nproc)
    n = 6000
    E = tb.b.xmax * 2.0 ** rng.uniform(-tb.b.k - 1.5, -1e-6, n)
    u = rng.random(n)
    proc, iv, rb = np.zeros(n, np.int32), np.zeros(n, np.int32), np.zeros(n)
    check(mp.ctx, lib().pt_debug_select(mp.ctx, 0, n, E.ctypes.data_as(C.POINTER(C.c_double)),
                                        u.ctypes.data_as(C.POINTER(C.c_double)), None,
                                        iv.ctypes.data_as(C.POINTER(C.c_int32)),
                                        proc.ctypes.data_as(C.POINTER(C.c_int32)),
                                        rb.ctypes.data_as(C.POINTER(C.c_double))))
    mp.close()
    i, t = tb.b.precheb(E)
    c = tb.rate[i]
    nu = (c[..., 0] * t[0][:, None] + c[..., 1] * t[1][:, None]) + c[..., 2] * t[2][:, None]
    want, xi = np.full(n, -1), u * rb
    margin = np.full(n, np.inf)
    scale = np.abs(nu).sum(axis=1)
    for j in range(nproc):
        open_ = want < 0
        # (a process of rate zero adds exactly nothing to either sum)
        near = np.where(nu[:, j] == 0.0, np.inf, np.abs(nu[:, j] - xi) / np.where(scale > 0.0, scale, 1.0))
        margin[open_] = np.fmin(margin, near)[open_]
        want[open_ & (nu[:, j] > xi)] = j
        xi = np.where(want < 0, xi - nu[:, j], xi)
    clear = ~(margin < 1e-12)
    assert clear.sum() > 0.99 * n
    assert np.array_equal(proc[clear], want[clear])
    if kind != "zeros" or nproc > 4:
        assert (want >= 0).any()
    assert (want < 0).any()


def test_a_row_that_is_not_a_number_does_not_reach_its_neighbours():
    """Photons whose rows are clean between rows of NaN: null collisions read past their row's
    end and must not be taken for an underestimated rate bound; in a NaN row they must."""
    te, tg, tp = H.tables()
    b = tg.b
    rate = np.zeros((b.k + 1, 4, 3))
    rate[1::2] = np.nan
    rb = np.zeros((1, b.k + 1, 3))
    rb[0, :, 0] = 1e13
    tb = ChebyshevCollisionTable([tg.proc[0]] * 4, b, rate, rb, tg.species, energy_cut=H.CUT)
    rows = np.arange(b.k + 1)
    mid = b.xmax * 2.0 ** (rows - b.k - 0.5)   # an energy inside each row (above the lowest)
    for odd in (0, 1):
        E = [e for q, e in zip(rows, mid) if q % 2 == odd and e > 2 * H.CUT][:3]
        mp = H.make_device(te, tb, tp, 5)
        soa = np.zeros((10, len(E)))
        soa[5] = np.array(E) / co.c
        soa[6] = 1.0
        soa[8] = 0.1
        mp.add_soa(1, soa, uid=np.arange(len(E), dtype=np.uint64))
        mp.init()
        if odd:
            with pytest.raises(Exception, match="rate bound"):
                mp.advance(1e-12)
        else:
            mp.advance(1e-12)
            assert mp.collision_counts(1)[0] > 0
        mp.close()
