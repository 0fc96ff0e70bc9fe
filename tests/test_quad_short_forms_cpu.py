"""The quotient and the square root that the quadcopter's step takes where no
operand is small or huge (an approximation within one unit in the last place,
then residuals) round correctly: the same operations on the CPU over a sweep of
operands, with every approximation that the unit may give."""
import numpy as np
import pytest

f32, f64 = np.float32, np.float64


def _ulp(x, k):
    return (x.view(np.int32) + np.int32(k)).view(f32)


def _fma(a, b, c):
    """a b + c rounded once: the product is exact in 64 bits, the sum is rounded
    to odd (its error by two-sum), which the rounding to 32 bits then keeps."""
    p, c = a.astype(f64) * b.astype(f64), c.astype(f64)
    s = p + c
    v = s - p
    err = (p - (s - v)) + (c - v)
    even = (s.view(np.int64) & 1) == 0
    s = np.where((err != 0) & even, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s)
    return s.astype(f32)


@pytest.mark.parametrize("off", [-1, 0, 1])
def test_root(off):
    # two binades of operands hold every mantissa of a root
    x = np.arange(0x3F800000, 0x40800000, 5, dtype=np.int64).astype(np.uint32).view(f32)
    want = np.sqrt(x.astype(f64)).astype(f32)  # (a root of a float is never a tie)
    s = _ulp(want, off)
    lo, hi = _ulp(s, -1), _ulp(s, 1)
    x64 = x.astype(f64)
    # residuals: signs of exact differences
    rl = x64 - lo.astype(f64) * s.astype(f64)
    rh = x64 - hi.astype(f64) * s.astype(f64)
    got = np.where(rh > 0, hi, np.where(rl <= 0, lo, s))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("off", [-1, 0, 1])
def test_quotient(off):
    """(A reciprocal one unit off is refined to the nearest float but for a
    divisor just below a power of two, where the step ends at a tie: there the
    unit gives the nearest float itself, which the device's test holds.)"""
    rng = np.random.default_rng(7 + off)
    n = 1 << 20
    edge = np.array([1.0, 1.0 + 2.0**-23, 1.5, 2.0 - 2.0**-23, 2.0 - 2.0**-22], f32)
    m = lambda: np.where(rng.random(n) < 0.1, rng.choice(edge, n),
                         (rng.integers(0, 1 << 23, n) + (127 << 23)).astype(np.uint32).view(f32)).astype(f32)
    b = np.ldexp(m(), rng.integers(-40, 0, n)).astype(f32)  # |cos theta|
    a = np.ldexp(m(), rng.integers(-40, 60, n)).astype(f32) * rng.choice(np.array([-1.0, 1.0], f32), n)
    y = _ulp((1.0 / b.astype(f64)).astype(f32), off)
    top = (b.view(np.uint32) & 0x7FFFFF) == 0x7FFFFF
    y = np.where(top, _ulp(y, -off), y).astype(f32)
    y = _fma(_fma(-b, y, np.ones(n, f32)), y, y)
    q = (a * y).astype(f32)
    q = _fma(_fma(-b, q, a), y, q)
    q = _fma(_fma(-b, q, a), y, q)
    want = (a / b).astype(f32)
    assert np.array_equal(q, want), np.flatnonzero(q != want)[:5]
