"""Reductions over a strided axis with few columns, or rows that no vector
width divides: lanes on several rows, the row's last vector drawn back over
its neighbour's columns, rows that start at any element, and splits whose
partials a second kernel combines (many rows), the last workgroup combines
(fewer) or that are not split."""
import numpy as np
import pytest

import macmetalpy_amd as cp

pytestmark = pytest.mark.gpu

COLS = [2, 3, 4, 5, 7, 8, 9, 15, 17, 31, 33, 50, 65, 127, 129, 255, 257, 511, 1001]
DTYPES = [np.float32, np.float64, np.float16, np.int16, np.int32, np.bool_]


def _data(g, shape, dt):
    if dt == np.bool_:
        return g.random(shape) < 0.5
    return g.integers(-20, 21, shape).astype(dt)  # sums exact in float64; ties


@pytest.mark.parametrize("rows", [3, 300, 5000, 40000])
@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: np.dtype(d).name)
def test_few_columns(rows, dt):
    g = np.random.default_rng(rows)
    for cols in COLS:
        if rows * cols > 6_000_000:
            continue
        h = _data(g, (rows, cols), dt)
        d = cp.array(h)
        for name in ("sum", "max", "min", "argmax", "argmin"):
            got, want = getattr(cp, name)(d, axis=0).get(), getattr(np, name)(h, axis=0)
            if name == "sum" and np.dtype(dt).kind == "f":
                want = np.sum(h.astype(np.float64), axis=0).astype(dt)
            assert got.dtype == want.dtype, (cols, name)
            assert np.array_equal(got, want), (cols, name)
    # an offset base (rows start at any element) and an outer extent above one
    h = _data(g, (4, rows // 3 + 1, 37), dt)
    d = cp.array(h)
    for f in (cp.sum, cp.max, cp.argmin):
        nf = getattr(np, f.__name__)
        want = nf(h.astype(np.float64) if f is cp.sum and np.dtype(dt).kind == "f" else h, axis=1)
        assert np.array_equal(f(d, axis=1).get(), want.astype(h.dtype) if f is not cp.argmin and
                              np.dtype(dt).kind == "f" else want)
        assert np.array_equal(f(d[1:], axis=1).get(), f(d, axis=1).get()[1:])


@pytest.mark.parametrize("rows,cols", [(50, 11), (3000, 6), (70000, 10), (70000, 131)])
def test_few_columns_nan(rows, cols):
    """NaN rules: max / argmax take the first NaN, the nan forms skip it."""
    g = np.random.default_rng(cols)
    h = g.standard_normal((rows, cols)).astype(np.float32)
    h[g.integers(0, rows, cols // 2), np.arange(cols // 2)] = np.nan
    d = cp.array(h)
    assert np.array_equal(cp.max(d, axis=0).get(), np.max(h, axis=0), equal_nan=True)
    assert np.array_equal(cp.argmax(d, axis=0).get(), np.argmax(h, axis=0))
    assert np.array_equal(cp.nanargmin(d, axis=0).get(), np.nanargmin(h, axis=0))
    assert np.array_equal(cp.nanmax(d, axis=0).get(), np.nanmax(h, axis=0))
    want = np.nanmean(h.astype(np.float64), axis=0)
    assert np.allclose(cp.nanmean(d, axis=0).get(), want, rtol=1e-6, atol=1e-7)
    inf = h.copy()
    inf[rows // 2] = -np.inf
    assert np.array_equal(cp.sum(cp.array(inf), axis=0).get(), np.sum(inf, axis=0), equal_nan=True)


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("outer,length,inner", [(5000, 20, 9), (9000, 60, 3), (4, 1, 700), (70, 16, 300),
                                                (70, 17, 301), (1, 2, 100_001), (40_000, 3, 2),
                                                (600, 15, 130), (3, 8, 4099)])
def test_short_axes(outer, length, inner, dt):
    """Axes of a few rows (a thread walks one by itself): every remainder of
    the row loop, whole and cut-off column vectors, rows shorter than one, an
    input that starts at any element; NaN and infinities."""
    g = np.random.default_rng(length)
    h = _data(g, (outer + 1, length, inner), dt)
    if np.dtype(dt).kind == "f":
        h[g.integers(0, outer, 20), g.integers(0, length, 20), g.integers(0, inner, 20)] = np.nan
        h[g.integers(0, outer, 20), g.integers(0, length, 20), g.integers(0, inner, 20)] = -np.inf
    d = cp.array(h)
    for x, y in ((d, h), (d[1:], h[1:])):
        for name in ("sum", "max", "min", "argmax", "argmin"):
            f, nf = getattr(cp, name), getattr(np, name)
            wide = name == "sum" and np.dtype(dt).kind == "f"
            want = nf(y.astype(np.float64) if wide else y, axis=1)
            want = want.astype(dt) if wide else want
            got = f(x, axis=1).get()
            assert got.dtype == want.dtype and np.array_equal(got, want, equal_nan=wide or
                                                              name in ("max", "min")), name
    if np.dtype(dt).kind == "f":
        assert np.array_equal(cp.nanmax(d, axis=1).get(), np.fmax.reduce(h, axis=1), equal_nan=True)


def test_partials_of_one_call_do_not_reach_the_next():
    """Reductions that leave raw partials for a second kernel, whose values
    are the numbers that calls are tagged with, between reductions that know
    their partials by the tag."""
    rows, cols = 400_000, 48
    raw = np.empty((rows, cols), np.int32)
    raw[:] = np.arange(cols * 8).reshape(8, cols)[np.arange(rows) % 8]
    big = np.random.default_rng(0).integers(-9, 9, (3000, 300)).astype(np.int32)
    draw, dbig = cp.array(raw), cp.array(big)
    flat = cp.array(big.ravel())
    for _ in range(40):
        assert np.array_equal(cp.max(draw, axis=0).get(), raw[7])
        assert np.array_equal(cp.argmax(draw, axis=0).get(), np.full(cols, 7))
        assert np.array_equal(cp.max(dbig, axis=0).get(), big.max(axis=0))
        assert np.array_equal(cp.sum(dbig, axis=0).get(), big.sum(axis=0))
        assert np.array_equal(cp.argmin(dbig, axis=0).get(), big.argmin(axis=0))
        assert int(cp.sum(flat)) == big.sum()
