"""The logarithm and the azimuth's sine and cosine of the step on the device, against values in
extended precision, through elastic collisions with injected uniforms: -log(u) is the new
particle's s, and a momentum along z is turned to p' = |p| (st cos, st sin, ...).

Tolerances: the logarithm is within 0.6 ulp by its construction (a table's two-part logarithm
and a polynomial, one rounding at the end).  The transverse components are two rounded
products with sine or cosine (within 0.8 ulp), together 1.8 ulp of each; their root sum of
squares, taken in extended precision, carries at most the larger of the two errors, so that
the quotient is within 3.6 ulp, here taken as 4."""
import ctypes as C

import numpy as np
import pytest

import helpers as H
from particulator_hip import co
from particulator_hip._lib import SOA, check, lib

pytestmark = pytest.mark.gpu

L = np.longdouble


def elastic(u):
    """the primaries after elastic collisions of 1 MeV electrons along z with uniforms u[i]"""
    te, tg, tp = H.tables()
    mp = H.make_device(te, tg, tp, 1, caps=(64, 64, 64))
    proc = next(j for j, p in enumerate(te.proc) if type(p).__name__ == "RelativisticCoulomb")
    u = np.ascontiguousarray(u, dtype=np.float64)
    n, stride = u.shape
    soa = np.zeros((10, n))
    soa[5] = 5e-22
    soa[6] = 1.0
    kind, draws = np.zeros(n, np.int32), np.zeros(n, np.int32)
    ost, osp, ouid = np.zeros((n, 3, 10)), np.zeros((n, 3), np.int32), np.zeros((n, 3), np.uint64)
    uid = np.arange(n, dtype=np.uint64)
    ip = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))
    dp = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    up = lambda a: a.ctypes.data_as(C.POINTER(C.c_uint64))
    check(mp.ctx, lib().pt_debug_collide(mp.ctx, 0, proc, n, SOA(*[dp(soa[f]) for f in range(10)]), up(uid), dp(u),
                                         stride, ip(kind), ip(draws), dp(ost), ip(osp), up(ouid)))
    mp.close()
    assert np.all(kind == 1) and np.all(draws == 4)
    return ost[:, 0]


def uniforms(n, azimuth=None, last=None):
    """azimuth, one accepted trial of the scattering angle, the draw of s"""
    u = np.full((n, 4), 0.5)
    u[:, 2] = 0.0  # accepted at once
    if azimuth is not None:
        u[:, 0] = azimuth
    if last is not None:
        u[:, 3] = last
    return u


def test_logarithm():
    rng = np.random.default_rng(3)
    u = np.concatenate([rng.random(200_000) + 2.0 ** -54, np.exp(-rng.uniform(0, 36, 100_000)),
                        1.0 - np.exp(-rng.uniform(0, 36, 100_000)), 2.0 ** -np.arange(1.0, 54.0),
                        [1.0 - 2.0 ** -53, 2.0 ** -53, 0.75, np.nextafter(0.75, 0), np.nextafter(0.75, 1)]])
    u = u[(u > 0) & (u < 1)]
    s = elastic(uniforms(u.size, last=u))[:, 8]
    want = -np.log(u.astype(L))
    ulp = np.spacing(np.abs(want.astype(np.float64))).astype(L)
    assert np.max(np.abs(s.astype(L) - want) / ulp) <= 0.6


def test_azimuth():
    rng = np.random.default_rng(4)
    k = np.arange(0, 9) / 8.0
    u = np.concatenate([rng.random(300_000), (k[:, None] + rng.choice([-1, 1], (9, 400)) * np.exp(
        -rng.uniform(2, 36, (9, 400)))).ravel(), k[:-1], [1.0 - 2.0 ** -53, 2.0 ** -53]])
    u = u[(u >= 0) & (u < 1)]
    st = elastic(uniforms(u.size, azimuth=u))
    phi = ((2.0 * np.pi) * u).astype(L)  # the device's product, rounded once
    x, y = st[:, 3].astype(L), st[:, 4].astype(L)
    T = np.sqrt(x * x + y * y)
    assert np.all(T > 0)
    for got, want in ((x / T, np.cos(phi)), (y / T, np.sin(phi))):
        # (np.longdouble's sine and cosine are good to 2^-63; beside their zeros what counts is
        # the argument, exact here)
        assert np.max(np.abs(got - want) / np.maximum(np.abs(want), L(2) ** -60)) <= 4 * 2.0 ** -53


def test_zero_draws_as_ieee_has_them():
    """An injected uniform of zero (a stream never yields one): no interval to the next
    collision is finite; the smallest numbers have theirs."""
    tiny = np.array([0.0, 5e-324, 1e-310, 2.3e-308])
    s = elastic(uniforms(tiny.size, last=tiny))[:, 8]
    assert s[0] == np.inf
    want = -np.log(tiny[1:].astype(L))
    assert np.allclose(s[1:].astype(L), want, rtol=1e-15, atol=0.0)
