"""The short quotient, reciprocal, square root and exponential of the FP64 kernels over the operand
ranges that they state: the correctly rounded results, bit for bit (the exponential: those of the
library's exp).  Significands: random ones, ones next to powers of two, exact quotients and squares."""
import numpy as np
import pytest

from lydion_amd import m1lya as M
from tests.helpers import bitdiff

pytestmark = pytest.mark.gpu

N = 200_000


def _significands(rng, n):
    """In [1, 2): a third random, a third within four steps of either end, a third short."""
    m = 1.0 + rng.integers(0, 1 << 52, n) * 2.0 ** -52
    steps = rng.integers(0, 4, n) * 2.0 ** -52
    ends = np.where(rng.random(n) < 0.5, 1.0 + steps, 2.0 - 2.0 ** -52 - steps)
    short = 1.0 + rng.integers(0, 1 << 12, n) * 2.0 ** -12
    kind = rng.integers(0, 3, n)
    return np.where(kind == 0, m, np.where(kind == 1, ends, short))


def _numbers(rng, lo, hi, n=N):
    """Significands at exponents lo .. hi - 1, both ends taken often."""
    e = np.where(rng.random(n) < 0.1, np.where(rng.random(n) < 0.5, lo, hi - 1), rng.integers(lo, hi, n))
    return np.ldexp(_significands(rng, n), e)


@pytest.mark.parametrize("d_lo,d_hi", [(-1000, 1000), (-2, 2), (-1000, -980), (795, 805)])
def test_quotient(d_lo, d_hi):
    rng = np.random.default_rng(11)
    d = _numbers(rng, d_lo, d_hi) * rng.choice([-1.0, 1.0], N)
    q = _numbers(rng, -999, 1000)
    with np.errstate(over="ignore", under="ignore"):
        near = d * q                                   # quotients next to q
        n = np.where(rng.random(N) < 0.5, near, _numbers(rng, -960, 1000))
        ok = np.isfinite(n) & (np.abs(n) >= 2.0 ** -960) & (np.abs(n) <= 2.0 ** 1000)
        want = n / d
        ok &= (np.abs(want) >= 2.0 ** -1000) & (np.abs(want) <= 2.0 ** 1000)
    n, d, want = n[ok], d[ok], want[ok]
    assert len(n) > N // 8
    assert bitdiff(M.selftest_math(4, n, d), want) == 0


def test_quotient_of_the_callers_divisors_and_zero():
    rng = np.random.default_rng(12)
    for d in (1e-300, 2.0 ** 800, 1.0 + 2.0 ** -52, 2.0 - 2.0 ** -52, 7.0, 5.0 + 2.0 * np.sqrt(2.0)):
        e = int(np.floor(np.log2(d)))
        n = _numbers(rng, max(-960, e - 999), min(1000, e + 999))
        assert bitdiff(M.selftest_math(4, n, np.full(N, d)), n / d) == 0, d
        zero = np.zeros(4)
        assert bitdiff(M.selftest_math(4, zero, np.full(4, d)), zero) == 0
    for n, d in ((np.inf, 3.0), (np.nan, 3.0), (1.0, np.nan), (1.0, np.inf)):
        assert np.isnan(M.selftest_math(4, np.full(4, n), np.full(4, d))).all()


@pytest.mark.parametrize("lo,hi", [(-1000, 1000), (-1, 1)])
def test_reciprocal(lo, hi):
    rng = np.random.default_rng(13)
    d = _numbers(rng, lo, hi) * rng.choice([-1.0, 1.0], N)
    assert bitdiff(M.selftest_math(5, d), 1.0 / d) == 0


@pytest.mark.parametrize("lo,hi", [(-700, 1000), (-1, 1)])
def test_root(lo, hi):
    rng = np.random.default_rng(14)
    x = _numbers(rng, lo, hi)
    m = _numbers(rng, lo // 2, hi // 2)
    square = m * m                                     # roots next to m
    x = np.where((rng.random(N) < 0.5) & (square >= 2.0 ** lo) & (square <= 2.0 ** hi), square, x)
    assert bitdiff(M.selftest_math(6, x), np.sqrt(x)) == 0


def test_exponential_is_the_librarys():
    rng = np.random.default_rng(15)
    x = np.concatenate([rng.uniform(-700, 700, N), rng.uniform(-1, 1, N), [0.0, -0.0, 700.0, -700.0, 1e-300, -1e-300]])
    assert bitdiff(M.selftest_math(7, x), M.selftest_math(2, x)) == 0
