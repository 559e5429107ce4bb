"""Which operands matmul reads where they lie (CPU), and the general float32 /
float64 kernel on extents around its tiles, K splits, transposed, strided and
misaligned operands against exact integer products (GPU)."""
import numpy as np
import pytest

import macmetalpy_amd as cp
from macmetalpy_amd import linalg_top


class _Strided:
    """Shape and element strides of a view, as the rule reads them."""

    def __init__(self, view):
        self._shape = view.shape
        self._strides = tuple(s // view.itemsize for s in view.strides)


def _views():
    x = np.arange(2 * 3 * 6 * 8, dtype=np.float32).reshape(2, 3, 6, 8)
    yield from (x, x.swapaxes(-1, -2), x[..., 1:], x[..., ::2], x[..., ::-1], x[:, ::2], x[::-1],
                x.transpose(1, 0, 2, 3), x.transpose(2, 0, 1, 3), x.transpose(3, 2, 1, 0),
                x[:1, :1], x[:1], x[:, :1, 2:, 3:], x[..., :1], x[..., :1, :], x[0, 0], x[0, 0].T,
                x[0, 0][::2], x[0, 0][:, 2:5].T, x[0].swapaxes(0, 1), x[..., 3:4].swapaxes(-1, -2))
    yield np.broadcast_to(x[0, 0], (2, 3, 6, 8))
    yield np.broadcast_to(x[0, 0, :1], (6, 8))
    yield np.broadcast_to(x[0, 0, :, :1], (6, 8))


def test_in_place_rule_addresses_every_element():
    """Wherever the rule accepts a view, (transposed, row stride, batch
    stride) gives the address of every element that the view's own strides
    give; what it refuses is copied as before."""
    taken = 0
    for v in _views():
        s = _Strided(v)
        got = linalg_top._in_place(s, v.shape[:-2])
        if got is None:
            continue
        taken += 1
        ta, ld, bs = got
        rows, cols = v.shape[-2:]
        assert ld >= (rows if ta else cols) and bs >= 0
        for b, idx in enumerate(np.ndindex(*v.shape[:-2])):
            for r in range(rows):
                for c in range(cols):
                    want = sum(i * t for i, t in zip(idx + (r, c), s._strides))
                    assert b * bs + (c * ld + r if ta else r * ld + c) == want
    assert taken >= 12


def test_in_place_rule_refuses():
    x = np.zeros((6, 8), np.float32)
    for v in (x[:, ::2], x[::-1], x[:, ::-1], np.broadcast_to(x[:1], (6, 8)),
              np.broadcast_to(x[:, :1], (6, 8))):
        assert linalg_top._in_place(_Strided(v), ()) is None
    y = np.zeros((4, 2, 6, 8), np.float32)
    assert linalg_top._in_place(_Strided(y.swapaxes(0, 1)), (2, 4)) is None
    assert linalg_top._in_place(_Strided(y[:, :1]), (4, 3)) is None  # broadcast batch


def _exact(a, b, got):
    want = np.matmul(a.astype(np.float64), b.astype(np.float64))
    assert got.shape == want.shape and np.array_equal(got.astype(np.float64), want)


def _ints(g, shape, dtype):
    return g.integers(-3, 4, shape).astype(dtype)


# Tile edges (32, 64, 128), slab edges (32 floats, 16 doubles), rows shorter
# than a vector, K splits (one long sum, uneven last range) and batches.
_SHAPES = [(1, 1, 2, 1), (1, 2, 2, 3), (1, 3, 5, 33), (1, 31, 33, 31), (1, 32, 32, 32),
           (1, 65, 63, 17), (1, 127, 129, 64), (1, 129, 257, 65), (1, 200, 130, 1000),
           (1, 2, 3, 40001), (1, 50, 70, 20000), (3, 33, 2, 35), (70, 20, 30, 40),
           (1, 1030, 700, 100), (1, 4100, 60, 50), (5, 128, 128, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch,m,n,k", _SHAPES)
def test_general_kernel_exact(batch, m, n, k, dtype):
    """Every combination of stored and transposed operands.  Integer values
    keep each sum exact, so the result equals the float64 product."""
    g = np.random.default_rng(m * 1000 + n + k)
    lead = (batch,) if batch > 1 else ()
    a, b = _ints(g, lead + (m, k), dtype), _ints(g, lead + (k, n), dtype)
    at, bt = np.ascontiguousarray(a.swapaxes(-1, -2)), np.ascontiguousarray(b.swapaxes(-1, -2))
    for x in (cp.array(a), cp.array(at).swapaxes(-1, -2)):
        for y in (cp.array(b), cp.array(bt).swapaxes(-1, -2)):
            _exact(a, b, cp.matmul(x, y).get())


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,n,k", _SHAPES + [(1, 64, 64, 5000), (1, 300, 1, 4000),
                                                   (1, 1, 300, 4000), (2, 640, 384, 448)])
def test_general_half_kernel_exact(batch, m, n, k):
    """float16: the same edges (slabs of 64, vectors of 8 and 4), contiguous
    and with row strides that leave rows on odd elements, NaN round the view.
    Sums of products of -1, 0 and 1 stay below 2048 here and so are exact."""
    g = np.random.default_rng(m * 1000 + n + k)
    lead = (batch,) if batch > 1 else ()
    a, b = (g.integers(-1, 2, lead + s).astype(np.float16) for s in ((m, k), (k, n)))
    want = np.matmul(a.astype(np.float32), b.astype(np.float32))
    assert np.abs(want).max() <= 2048
    got = cp.matmul(cp.array(a), cp.array(b)).get()
    assert got.dtype == np.float16 and np.array_equal(got.astype(np.float32), want)
    if batch == 1:
        from macmetalpy_amd._backend import HipBackend
        from macmetalpy_amd._dtypes import dtype_code
        pa, pb = np.full((m, k + 3), np.nan, np.float16), np.full((k, n + 5), np.nan, np.float16)
        pa[:, :k], pb[:, :n] = a, b
        c = np.full((m, n + 1), 7.0, np.float16)
        da, db, dc = (cp.array(x)._ensure_gpu() for x in (pa, pb, c))
        HipBackend().matmul(dtype_code(np.dtype(np.float16)), 1, m, n, k, da._ptr, k + 3, 0, db._ptr,
                            n + 5, 0, dc._ptr, n + 1, 0)
        out = dc.get()
        assert np.array_equal(out[:, :n].astype(np.float32), want) and np.all(out[:, n:] == 7.0)


def _to_bf16(x):
    """Bits of the bfloat16 values of ``x``, which are exact there."""
    bits = np.ascontiguousarray(x, np.float32).view(np.uint32)
    assert not np.any(bits & 0xFFFF)
    return (bits >> 16).astype(np.uint16)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,m,n,k", [(1, 1, 2, 1), (1, 65, 63, 17), (1, 129, 257, 65), (1, 64, 64, 5000),
                                         (70, 20, 30, 40), (1, 1030, 700, 100), (1, 300, 1, 4000),
                                         (2, 640, 384, 448), (1, 2304, 2304, 64), (8, 1024, 1024, 128)])
def test_bfloat16_products_exact(batch, m, n, k):
    """bfloat16 has no NumPy type: its products through the entry point, all
    kernels of the 16-bit types (general, whole aligned tiles, 256 wide tiles).
    Products of -1, 0 and 1 over at most 200 terms are exact in eight bits."""
    from macmetalpy_amd._backend import HipBackend
    g = np.random.default_rng(m + n + k)
    a, b = g.integers(-1, 2, (batch, m, k)), g.integers(-1, 2, (batch, k, n))
    b[:, 200:] = 0
    da, db = (cp.array(_to_bf16(x))._ensure_gpu() for x in (a, b))
    c = cp.array(np.full((batch, m, n), 7, np.uint16))._ensure_gpu()
    HipBackend().matmul(10, batch, m, n, k, da._ptr, k, m * k, db._ptr, n, k * n, c._ptr, n, m * n)
    want = np.matmul(a.astype(np.float32), b.astype(np.float32))
    assert np.array_equal(c.get(), _to_bf16(want))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.float16])
def test_rows_too_far_apart_for_lane_offsets(dtype):
    """Row strides of 2^24 elements and more take the guarded loads: as the
    left and the right operand, as stored and transposed."""
    from macmetalpy_amd._backend import HipBackend
    from macmetalpy_amd._dtypes import dtype_code
    g = np.random.default_rng(9)
    ld, rows, cols = (1 << 24) + 5, 5, 150
    a = _ints(g, (rows, cols), dtype)
    big = cp.zeros((rows, ld), dtype=dtype)
    v = big[:, 3:3 + cols]
    v[...] = cp.array(a)
    x, y = _ints(g, (cols, 70), dtype), _ints(g, (rows, 40), dtype)
    _exact(a, x, cp.matmul(v, cp.array(x)).get())
    _exact(a.T, y, cp.matmul(v.T, cp.array(y)).get())
    _exact(x.T, a.T, cp.matmul(cp.array(x).T, v.T).get())
    _exact(y.T, a, cp.matmul(cp.array(y).T, v).get())
    be, dc = HipBackend(), dtype_code(np.dtype(dtype))  # copies are Python's: the strides themselves
    dx, dy = cp.array(x)._ensure_gpu(), cp.array(np.ascontiguousarray(y.T))._ensure_gpu()
    c = cp.array(np.zeros((rows, 70), dtype))._ensure_gpu()
    be.matmul(dc, 1, rows, 70, cols, v._ptr, ld, 0, dx._ptr, 70, 0, c._ptr, 70, 0)
    _exact(a, x, c.get())
    c = cp.array(np.zeros((40, cols), dtype))._ensure_gpu()
    be.matmul(dc, 1, 40, cols, rows, dy._ptr, rows, 0, v._ptr, ld, 0, c._ptr, cols, 0)
    _exact(y.T, a, c.get())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_general_kernel_views(dtype):
    """Row slices, column slices (misaligned rows), steps, reversed and
    broadcast operands, and batches that do and do not nest.  The memory
    round the views holds NaN, which must not reach a result."""
    g = np.random.default_rng(7)
    big = np.full((4, 3, 70, 90), np.nan, dtype)
    big[:, :, 3:67, 5:82] = _ints(g, (4, 3, 64, 77), dtype)
    w = np.full((90, 50), np.nan, dtype)
    w[2:79, 1:42] = _ints(g, (77, 41), dtype)
    dbig, dw = cp.array(big), cp.array(w)
    pick = [lambda x: x[0, 0], lambda x: x[:, 0], lambda x: x[0], lambda x: x,
            lambda x: x.transpose(1, 0, 2, 3), lambda x: x[::2, 1:]]
    for f in pick:
        a, da = f(big)[..., 3:67, 5:82], f(dbig)[..., 3:67, 5:82]
        b, db = w[2:79, 1:42], dw[2:79, 1:42]
        _exact(a, b, cp.matmul(da, db).get())
        at, dat = a.swapaxes(-1, -2), da.swapaxes(-1, -2)
        _exact(b.T, at, cp.matmul(db.T, dat).get())
        _exact(at, a, cp.matmul(dat, da).get())
    a, da = big[0, 0, 3:67, 5:82], dbig[0, 0, 3:67, 5:82]
    _exact(a[::2], w[2:79, 1:42], cp.matmul(da[::2], dw[2:79, 1:42]).get())
    _exact(a[:, ::-1], w[2:79, 1:42], cp.matmul(da[:, ::-1], dw[2:79, 1:42]).get())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(40, 30, 60000), (4, 4, 2_000_003), (128, 128, 16384)])
def test_long_sums_are_cut(m, n, k):
    """At most 128 x 128 outputs over 16,384 terms or more: ranges of at most
    2048 terms, added in float64, so a float32 sum's error stays below 2049
    roundings of |A| |B| plus the result's own."""
    g = np.random.default_rng(3)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    got = cp.matmul(cp.array(a), cp.array(b)).get().astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(got - a @ b) <= 2050 * 2.0 ** -24 * (np.abs(a) @ np.abs(b)))
