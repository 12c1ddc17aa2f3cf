"""The softmax's division by one shared reciprocal (divide_all, dcrf_device.h) in host
arithmetic, over its operands 0 <= y <= 1 <= s <= 1024: the rounded quotient for y >= 2^-100,
whose residual no operand leaves inexact, and one unit in the last place for smaller y
(subnormal ones and subnormal quotients too), with the hardware's reciprocal exact or one
unit off either way."""
import numpy as np
import pytest

f32, wide = np.float32, np.longdouble
pytestmark = pytest.mark.skipif(np.finfo(wide).nmant < 63, reason="needs a 64-bit significand")


def fma(a, b, c):
    return (a.astype(wide) * b.astype(wide) + c.astype(wide)).astype(f32)


def divide_all(y, s, rcp):
    rc = fma(fma(-s, rcp, np.ones_like(s)), rcp, rcp)
    a = y * rc
    return fma(fma(-s, a, y), rc, a)


@pytest.mark.parametrize("lo,hi,ulps", [(-100, 0, 0), (-126, -100, 1), (-149, -120, 1)])
@pytest.mark.parametrize("off", [-1, 0, 1])
def test_quotient(lo, hi, ulps, off):
    rng = np.random.default_rng(-lo)
    n = 300_000
    s = np.exp2(rng.uniform(0, 10, n)).astype(f32)
    s[:4096] = np.tile(np.arange(1, 1025), 4)
    y = np.exp2(rng.uniform(lo, hi, n)).astype(f32)
    y[::1000] = min(1.0, 2.0 ** hi)
    r = (1 / s.astype(np.float64)).astype(f32)
    rcp = r if off == 0 else np.nextafter(r, f32(0) if off < 0 else f32(2))
    got, want = divide_all(y, s, rcp), y / s  # (numpy's division is correctly rounded)
    d = np.abs(got.view(np.int32).astype(np.int64) - want.view(np.int32))
    assert d.max() <= ulps


def test_edges():
    one = np.ones(3, f32)
    y = np.array([0.0, 1.0, np.nan], f32)
    assert np.array_equal(divide_all(y, one, one), y, equal_nan=True)
    assert np.isnan(divide_all(np.ones(1, f32), np.full(1, np.nan, f32), np.full(1, np.nan, f32))).all()
