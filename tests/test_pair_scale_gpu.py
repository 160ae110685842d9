"""The force's pair scale (short exact root, reciprocal and quotient) against
the general IEEE sequences on the device, and those against numpy: bit for
bit wherever the step would keep the short form (its range check holds), and
the range check itself on both sides of its bounds."""
import ctypes as C

import numpy as np
import pytest

from pibiti_amd import sph

pytestmark = pytest.mark.gpu

ONE = np.float32(1.0)


def pairs(par, r2, psum, rr):
    """(fast, general, in_range) of the pairs; scalars are repeated."""
    r2, psum, rr = (np.ascontiguousarray(x) for x in np.broadcast_arrays(*(np.asarray(x, np.float32)
                                                                           for x in (r2, psum, rr))))
    n = r2.size
    fast, general = np.empty((n, 2), np.float32), np.empty((n, 2), np.float32)
    ok = np.empty(n, np.uint32)
    par = np.asarray(par, np.float32)
    f = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))
    st = sph.lib().sph_pair_selftest(n, f(par), f(r2), f(psum), f(rr), f(fast), f(general),
                                     ok.ctypes.data_as(C.POINTER(C.c_uint32)))
    assert st == sph.SPH_OK, sph.strerror(st)
    return fast, general, ok.astype(bool)


def same(a, b):
    return (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))


def check(par, r2, psum, rr, least=1.0):
    """Where the short form is kept it is the general one; it is kept for at
    least that share of the pairs."""
    fast, general, ok = pairs(par, r2, psum, rr)
    bad = np.flatnonzero(ok & ~same(fast, general).all(axis=1))
    assert bad.size == 0, (bad.size, bad[:3], fast[bad[:3]], general[bad[:3]])
    assert ok.mean() >= least, ok.mean()
    return general


def mantissas(exponent):
    return (np.arange(2 ** 23, dtype=np.uint32) | np.uint32((127 + exponent) << 23)).view(np.float32)


# h = 0, minDens = 1 and a tiny rr make the kernel-density product -r
@pytest.mark.parametrize("exponent", [0, 1, -59, 94])
def test_every_root(exponent):
    print("case: roots, exponent", exponent, flush=True)
    x = mantissas(exponent)
    g = check((0.0, 1.0, 0.0, 1.0), x, ONE, np.float32(2.0 ** -40))
    assert np.array_equal(-g[:, 1], np.sqrt(x))


# h = 0 and r = 1: the kernel-density product is -1 / rr
@pytest.mark.parametrize("exponent", [0, -60, 95])
def test_every_reciprocal(exponent):
    print("case: reciprocals, exponent", exponent, flush=True)
    x = mantissas(exponent)
    g = check((0.0, 1.0, 0.0, 2.0 ** 126), ONE, ONE, x)
    assert np.array_equal(-g[:, 1], ONE / x)


def near_boundary(rng, count):
    """(a, b): integers of 24 bits whose quotient lies within 7 units of the
    product's last place of the middle between two floats: with the middle
    m / 2, m odd, a 2^k - b m = d for a small d."""
    out = []
    b0 = rng.integers(2 ** 22, 2 ** 23, count).astype(np.uint64) * np.uint64(2) + np.uint64(1)
    inv = b0.copy()  # b^-1 modulo 2^64 by Newton's iteration
    for _ in range(6):
        inv = inv * (np.uint64(2) - b0 * inv)
    for d in (-7, -5, -3, -1, 1, 3, 5, 7):
        for k in (24, 25):
            mod = np.uint64(2 ** k - 1)
            m = inv * np.uint64(-d & (2 ** 64 - 1)) & mod
            if k == 24:
                m = m | np.uint64(2 ** 24)
            num = (b0 * m).astype(np.int64) + d
            a = num >> k
            keep = (num & (2 ** k - 1)) == 0
            keep &= (m >= 2 ** 24) & (m < 2 ** 25) & (m & np.uint64(1) == 1) & (a >= 2 ** 23) & (a < 2 ** 24)
            out.append(np.stack([a[keep], b0[keep].astype(np.int64)], axis=1))
    return np.concatenate(out)


# h = 1 and r < 2^-26: h - r rounds to 1, so a = psum and the term is a / r
@pytest.mark.parametrize("exponent", [0, 94, -59])
def test_quotients_near_rounding_boundaries(exponent):
    rng = np.random.default_rng(11)
    ab = near_boundary(rng, 500_000)
    extra = rng.integers(2 ** 23, 2 ** 24, (2_000_000, 2))
    for what, q in (("near boundaries", ab), ("random", extra)):
        print("case:", len(q), "quotients", what, flush=True)
        a = np.ldexp(q[:, 0].astype(np.float32), exponent - 23)
        r = np.ldexp(q[:, 1].astype(np.float32), -27 - 23)
        r2 = (r * r).astype(np.float32)
        assert np.array_equal(np.sqrt(r2), r)  # the root of a rounded square
        g = check((1.0, 1.0, 0.0, 1.0), r2, a, ONE)
        assert np.array_equal(g[:, 0], a / r)
    assert len(ab) > 1_000_000


EDGES = np.array([0.0, 1e-45, 2.0 ** -126, 2.0 ** -91, 2.0 ** -90, 2.0 ** -61, np.nextafter(2.0 ** -60, 0, dtype=np.float32),
                  2.0 ** -60, 2.0 ** -30, 1.0, 2.0 ** 60, 1.5 * 2.0 ** 95, np.nextafter(2.0 ** 96, 0, dtype=np.float32),
                  2.0 ** 96, 2.0 ** 127, np.inf, np.nan], np.float32)


@pytest.mark.parametrize("min_dist", [0.0, 1e-45, 2.0 ** -31, 0.005, 2.0 ** 49, np.inf, np.nan])
@pytest.mark.parametrize("min_dens", [1e-6, 2.0 ** 126, 2.0 ** 127, np.inf, np.nan])
def test_edges_of_the_range(min_dist, min_dens):
    """Every combination of operands around the bounds, h from tiny to huge:
    infinities, zeros, NaN and denormals included."""
    e = np.concatenate([EDGES, -EDGES])
    r2, psum, rr = (x.ravel() for x in np.meshgrid(EDGES, e, e, indexing="ij"))
    for h in (0.02, 1.0, 2.0 ** 50, 2.0 ** 100):
        for spiky in (-1.0, -2.0 ** 38):
            check((h, spiky, min_dist, min_dens), r2, psum, rr, least=0.0)


def test_a_quotient_beyond_the_largest_float():
    """|a| = 1.5 2^95 over r = 1.25 2^-44 overflows: infinite, not NaN."""
    r2 = np.float32((1.25 * 2.0 ** -44) ** 2)
    g = check((1.0, 1.5, 0.0, 1.0), r2.reshape(1), np.float32(2.0 ** 95), ONE, least=0.0)
    assert np.isinf(g[0, 0])


def test_ordinary_pairs_stay_in_range():
    rng = np.random.default_rng(12)
    n = 1_000_000
    h = 0.02
    r2 = (h * rng.random(n) ** (1 / 3)).astype(np.float32) ** 2
    par = (h, -45.0 / (np.pi * h ** 6), 0.005, 1e-6)
    check(par, r2, rng.normal(0, 3000, n).astype(np.float32), rng.uniform(1e5, 4e6, n).astype(np.float32), least=0.999)


def test_pairs_without_pressure_stay_in_range():
    """Stiffness 0: the pressure sum is a zero of either sign."""
    rng = np.random.default_rng(13)
    n, h = 100_000, 0.02
    r2 = (h * rng.random(n) ** (1 / 3)).astype(np.float32) ** 2
    zero = np.where(rng.random(n) < 0.5, np.float32(0.0), np.float32(-0.0)).astype(np.float32)
    for spiky in (-45.0 / (np.pi * h ** 6), 45.0 / (np.pi * h ** 6)):
        g = check((h, spiky, 0.005, 1e-6), r2, zero, rng.uniform(1e5, 4e6, n).astype(np.float32), least=0.999)
        assert not np.any(g[:, 0])
