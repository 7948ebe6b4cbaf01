"""The kernels' short exact forms of roots, reciprocals and quotients
(pathmath.hpp) against IEEE single precision, bit for bit: every significand
where that is the whole argument (a power of two, for a root a power of four,
scales operand and result alike), both sides of each guard, and quotients next
to a rounding boundary."""
import numpy as np
import pytest

import raydar_amd as ra

pytestmark = pytest.mark.gpu

EDGES = [2.0 ** -149, 2.0 ** -126, 2.0 ** -97, 2.0 ** -96, 2.0 ** -60, 2.0 ** -48, 2.0 ** -20, 0.5, 1.0, 2.0 ** 20,
         2.0 ** 59, 2.0 ** 60, 2.0 ** 95, 2.0 ** 96, 2.0 ** 99, 2.0 ** 100, 2.0 ** 127]


def _same(got, want):
    # (a NaN's bits are the machine's own)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    np.testing.assert_array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))


def _around(values):
    v = np.array(values, np.float32).view(np.uint32).astype(np.int64)
    v = (v[:, None] + np.arange(-3, 4)).ravel()
    v = v[(v >= 0) & (v <= 0x7f800000)].astype(np.uint32).view(np.float32)
    return np.concatenate([v, -v, np.array([0.0, -0.0, np.inf, -np.inf, np.nan], np.float32)])


def _octave(exponent):
    return (np.arange(1 << 23, dtype=np.uint32) | np.uint32((exponent + 127) << 23)).view(np.float32)


@pytest.mark.parametrize("which", ["sqrt", "sqrt_normal"])
@pytest.mark.parametrize("exponent", [-96, 0, 1, 99])
def test_roots_of_every_significand(which, exponent):
    x = _octave(exponent)
    _same(ra.debug_arith(which, x), np.sqrt(x))


@pytest.mark.parametrize("which", ["rcp", "rcp_normal"])
@pytest.mark.parametrize("exponent", [-60, 0, 59])
def test_reciprocals_of_every_significand(which, exponent):
    x = _octave(exponent)
    _same(ra.debug_arith(which, x), np.float32(1) / x)
    _same(ra.debug_arith(which, -x), np.float32(1) / -x)


def test_roots_and_reciprocals_at_their_guards():
    x = _around(EDGES)
    with np.errstate(all="ignore"):
        _same(ra.debug_arith("sqrt", x), np.sqrt(x))
        _same(ra.debug_arith("rcp", x), np.float32(1) / x)


def test_normalised_vectors():
    rng = np.random.default_rng(5)
    x, y = (np.ldexp(rng.uniform(-1, 1, 1 << 20), rng.integers(-50, 50, 1 << 20)).astype(np.float32)
            for _ in range(2))
    e = _around(EDGES)
    a, b = np.concatenate([x, e, e]), np.concatenate([y, e, np.zeros_like(e)])
    with np.errstate(all="ignore"):
        q = a * a + b * b + np.float32(0)
        _same(ra.debug_arith("unit", a, b), a * (np.float32(1) / np.sqrt(q)))


@pytest.mark.parametrize("seed", range(3))
def test_quotients_next_to_a_rounding_boundary(seed):
    # a quotient's exact value n / a lies close to the middle of two floats if n
    # is the float next to a times that middle
    rng = np.random.default_rng(seed)
    m = 1 << 21
    a = ((rng.integers(0, 1 << 23, m) | (127 << 23)).astype(np.uint32)).view(np.float32)
    middle = 1.0 + (2 * rng.integers(0, 1 << 23, m) + 1) * 2.0 ** -24
    n = (a.astype(np.float64) * middle).astype(np.float32)
    n = (n.view(np.uint32)[None, :] + np.arange(-1, 2, dtype=np.int64)[:, None]).astype(np.uint32).view(np.float32)
    n = n.ravel()
    a = np.tile(a, 3)
    # anywhere in the ranges that the form is for
    n = np.ldexp(n, rng.integers(-60, 58, n.size)).astype(np.float32) * rng.choice([-1, 1], n.size).astype(np.float32)
    a = np.ldexp(a, rng.integers(-20, 20, a.size)).astype(np.float32) * rng.choice([-1, 1], a.size).astype(np.float32)
    _same(ra.debug_arith("div", n, a), n / a)
