"""Scans of short rows, row tails and odd columns: row lengths around a lane's
vector, a wave's step and a tile, row counts on both sides of each choice of
waves per row, rows that start at any element, and strided scans whose column
count no vector divides."""
import numpy as np
import pytest

import macmetalpy_amd as cp

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.float16, np.int16, np.int32, np.int64, np.uint16, np.bool_]


def _data(g, shape, dt):
    return (g.integers(0, 2, shape) if dt == np.bool_ else g.integers(0, 3, shape) if dt == np.uint16
            else g.integers(-1, 2, shape)).astype(dt)


def _check(h, axis):
    """Sums of small integers are exact in every type here."""
    got, want = cp.cumsum(cp.array(h), axis=axis).get(), np.cumsum(h.astype(np.int64), axis=axis)
    assert got.dtype == np.cumsum(h[:1], axis=axis).dtype
    assert np.array_equal(got.astype(np.int64), want)


@pytest.mark.parametrize("rows", [1, 3, 600, 2100])
@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: np.dtype(d).name)
def test_short_rows(rows, dt):
    g = np.random.default_rng(rows)
    for n in (1, 2, 7, 8, 9, 63, 64, 255, 256, 257, 511, 513, 1023, 2049, 4100, 8191, 8193, 16383,
              16384, 16385, 20001, 33000):
        if rows * n > 2_200_000 or (dt == np.float16 and n > 2000):
            continue
        _check(_data(g, (rows, n), dt), 1)


@pytest.mark.parametrize("dt", [np.float32, np.int32], ids=lambda d: np.dtype(d).name)
def test_unaligned_long_rows(dt):
    """Rows longer than a tile that start at odd elements, many and few."""
    g = np.random.default_rng(1)
    for rows, n in ((300, 17001), (5, 40003), (257, 16387)):
        _check(_data(g, (rows, n), dt), 1)
    h = _data(g, 70001, dt)
    d = cp.array(h)
    assert np.array_equal(cp.cumsum(d[1:]).get().astype(np.int64), np.cumsum(h[1:].astype(np.int64)))


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.float16, np.int32, np.int16],
                         ids=lambda d: np.dtype(d).name)
def test_odd_columns(dt):
    g = np.random.default_rng(2)
    for rows, cols in ((1, 5), (63, 9), (700, 1023), (1500, 7), (1500, 17), (130, 2051), (2000, 3),
                       (3000, 4), (3001, 7), (9000, 33), (3000, 1023), (8200, 37)):
        _check(_data(g, (rows, cols), dt), 0)
    h = _data(g, (3, 200, 33), dt)
    _check(h, 1)
    d = cp.array(h)
    assert np.array_equal(cp.cumsum(d[1:], axis=1).get(), cp.cumsum(d, axis=1).get()[1:])


def test_float_rows_round_once_and_repeat():
    """float32 rows accumulate in float64 (within one rounding of its own
    sums), give the same bits again, and pass infinities and NaN on."""
    g = np.random.default_rng(3)
    for rows, n in ((1, 9000), (40, 5000), (3000, 700)):
        h = g.standard_normal((rows, n), dtype=np.float32)
        d = cp.array(h)
        got = cp.cumsum(d, axis=1).get()
        ref = np.cumsum(h.astype(np.float64), axis=1)
        bound = 2.0 ** -24 * np.abs(ref) + n * 2.0 ** -52 * np.cumsum(np.abs(h).astype(np.float64), axis=1)
        assert np.all(np.abs(got - ref) <= bound)
        assert np.array_equal(got, cp.cumsum(d, axis=1).get())
    h = np.ones((3, 1000), np.float32)
    h[0, 300], h[1, 400], h[1, 500], h[2, 700] = np.inf, np.inf, -np.inf, np.nan
    assert np.array_equal(cp.cumsum(cp.array(h), axis=1).get(), np.cumsum(h, axis=1), equal_nan=True)
    p = np.full((5, 900), 2.0, np.float32)
    p[1] = 0.5
    assert np.array_equal(cp.cumprod(cp.array(p), axis=1).get(),
                          np.cumprod(p.astype(np.float64), axis=1).astype(np.float32))
