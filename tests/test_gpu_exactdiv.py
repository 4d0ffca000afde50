"""The quotients and roots by refined estimates (m2c_exactdiv.h) against IEEE
division and square root, bit for bit, over the ranges its header states:
random operands over all exponents, denominators whose reciprocal is nearest
to the middle of two doubles (significands of ones, Markstein's exception),
quotients nearest to such a middle, and numerators of zero."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libexactdiv.so")
N = 1 << 21


@pytest.fixture(scope="module")
def device():
    from m2c_amd import runtime
    runtime.lib()
    L = C.CDLL(LIB)
    p = C.POINTER(C.c_double)

    def run(a, b=None):
        a = np.ascontiguousarray(a)
        b = None if b is None else np.ascontiguousarray(b)
        out = np.empty_like(a)
        ptr = lambda x: None if x is None else x.ctypes.data_as(p)  # noqa: E731
        assert L.exactdiv(ptr(a), ptr(b), ptr(out), C.c_int(a.size)) == 0
        return out

    return run


def _numbers(rng, n, lo, hi):
    """Random significands and signs, exponents uniform in [lo, hi)."""
    return np.ldexp(rng.choice([-1.0, 1.0], n) * rng.uniform(1.0, 2.0, n), rng.integers(lo, hi, n))


def _same(x, y):
    bad = np.nonzero(x.view(np.int64) != y.view(np.int64))[0]
    assert bad.size == 0, (bad.size, bad[:4], x[bad[:4]], y[bad[:4]])


@pytest.mark.parametrize("seed", range(4))
def test_random_quotients(device, seed):
    rng = np.random.default_rng(seed)
    b = _numbers(rng, N, -900, 900)
    with np.errstate(over="ignore", under="ignore"):
        a = (_numbers(rng, N, -900, 1000) if seed % 2 else
             np.ldexp(b, rng.integers(-900, 900, N)) * rng.uniform(0.5, 2.0, N))
        q = a / b
    keep = (np.abs(a) >= 2.0**-900) & (np.abs(a) <= 2.0**1000) & (np.abs(q) >= 2.0**-1000) & (np.abs(q) <= 2.0**1000)
    assert keep.sum() > N // 4
    _same(device(a[keep], b[keep]), q[keep])


def test_denominators_with_reciprocals_between_two_doubles(device):
    rng = np.random.default_rng(5)
    b = (2.0**53 - rng.integers(1, 200, N)) * np.ldexp(1.0, rng.integers(-500, 500, N))
    a = _numbers(rng, N, -400, 400)
    a[::3] = 2.0**53 - rng.integers(0, 200, a[::3].size)
    _same(device(a, b), a / b)


@pytest.mark.parametrize("side", [-1, 1])
def test_quotients_nearest_to_the_middle_of_two_doubles(device, side):
    """a / b = M / 2^54 + side / (2^54 b) with M odd, of 54 bits."""
    rng = np.random.default_rng(7 + side)
    a, b = [], []
    for v in rng.integers(2**51, 2**52, 30000):
        den = 2 * int(v) + 1
        m = -side * pow(den, -1, 2**54) % 2**54  # den m = -side mod 2^54
        if m >= 2**53:
            a.append((den * m + side) // 2**54)
            b.append(den)
    assert len(a) > 10000 and max(a) < 2**53
    a, b = np.array(a, dtype=np.float64), np.array(b, dtype=np.float64)
    s = np.ldexp(1.0, rng.integers(-400, 400, a.size))
    t = np.ldexp(1.0, rng.integers(-400, 400, a.size))
    _same(device(a * s, b * t), (a * s) / (b * t))


def test_zero_numerators(device):
    b = _numbers(np.random.default_rng(9), 4096, -900, 900)
    assert np.all(device(np.zeros(4096), b) == 0.0)


@pytest.mark.parametrize("seed", range(2))
def test_random_roots(device, seed):
    x = np.abs(_numbers(np.random.default_rng(seed), N, -700, 900))
    _same(device(x), np.sqrt(x))


def test_roots_nearest_to_the_middle_of_two_doubles(device):
    """Of doubles next to the square of such a middle, the nearest ones."""
    rng = np.random.default_rng(3)
    x = []
    for m in rng.integers(2**53, 2**54, 300000):
        sq = (2 * (int(m) // 2) + 1) ** 2  # 107 or 108 bits: the square of an odd 54-bit number
        shift = sq.bit_length() - 53
        low = sq & ((1 << shift) - 1)
        if min(low, (1 << shift) - low) < 1 << (shift - 6):
            x.append(((sq >> shift) + (low >> (shift - 1)), shift - 106))
    assert len(x) > 5000
    v = np.array([float(q) for q, _ in x]) * np.array([2.0**e for _, e in x])
    v = np.concatenate([v * 4.0**k for k in (-300, -7, 0, 11, 300)])
    _same(device(v), np.sqrt(v))
