"""The flat launch of fused expressions (rows too short or too odd to be a
workgroup's): its leaf classes and generated source on the CPU, and its
results on the GPU against NumPy and the op-by-op evaluation."""
import itertools

import numpy as np
import pytest

import macmetalpy_amd as cp
from macmetalpy_amd import _fusion as F
from macmetalpy_amd._backend import DeviceBuffer, rtc_build


def _leaf(shape, dtype, strides, ptr):
    return F.InputNode(DeviceBuffer(ptr, 0, owned=False), shape, dtype, strides)


def _plan(leaves, shape, dtype=np.float32):
    root = leaves[0]
    for x in leaves[1:]:
        root = F.BinaryOpNode("add_op", root, x, shape, dtype)
    prog = F._Program(root)
    cshape, outer, cols, leaf_str, kinds = F._plan(prog, shape, False)
    flat = F._flat_kinds(outer, cols, leaf_str, [F._leaf_ptr(a) for a in prog.arrays],
                         [a._dtype.itemsize for a in prog.arrays], 0x20000, 4, F._map_tile(kinds))
    return prog, outer, cols, leaf_str, flat


# (strides of a leaf over (rows, cols), rows x cols -> its class or None)
def _strides(cols):
    return {"full": (cols, 1), "row": (0, 1), "column": (1, 0), "columns": (5, 0),
            "padded": (cols + 4, 1), "odd pad": (cols + 3, 1), "transposed": (1, 7),
            "stepped": (2 * cols, 2), "reversed": (cols, -1), "one": (0, 0)}


@pytest.mark.parametrize("cols", [1, 2, 3, 4, 7, 50, 64, 255, 256, 257, 1000, 4095, 4096, 4097, 8192])
def test_leaf_classes_address_every_element(cols):
    """Each class stands for the leaf's own strides, vectors are aligned, and
    rows of whole tiles (or too long for spread loads) stay with the row
    launch."""
    rows = 70000
    for name, st in _strides(cols).items():
        for ptr in (0x10000, 0x10004):
            x = _leaf((rows, cols), np.float32, (cols, 1), 0x40000)
            y = _leaf((rows, cols), np.float32, st, ptr)
            _, outer, c, leaf_str, flat = _plan([x, y], (rows, cols))
            if len(outer) != 1:
                assert flat is None  # both contiguous: one flat row already
                continue
            if c % 4 == 0 and c >= 4096:
                assert flat is None
                continue
            if flat is None:
                assert c >= 256
                continue
            (rs, cs), kind = leaf_str[1], flat[1]
            want = {"f": (c, 1), "q": (0, 1), "p": (0, 1), "w": (rs, 0), "r": (rs, 0),
                    "v": (rs, 1), "g": (rs, cs)}[kind]
            assert (rs, cs) == want, (name, kind)
            if kind in "fqv":
                assert ptr % 16 == 0
            if kind in "qwv":
                assert c % 4 == 0
            if kind == "v":
                assert rs % 4 == 0
    big = _leaf((1 << 21, 1024), np.float32, (1024, 1), 0x40000)
    row = _leaf((1 << 21, 1024), np.float32, (0, 1), 0x10000)
    assert _plan([big, row], (1 << 21, 1024))[-1] is None  # 2^31 elements
    small = _leaf((600, 100), np.float32, (100, 1), 0x40000)
    srow = _leaf((600, 100), np.float32, (0, 1), 0x10000)
    assert _plan([small, srow], (600, 100))[-1] is None  # under 2^16 elements


@pytest.mark.parametrize("out", [np.float32, np.float16, np.float64, np.bool_, np.int64])
def test_flat_source_compiles(out):
    kinds = ["f", "p", "q", "r", "w", "v", "g"]
    leaves = [_leaf((9, 8), out, (8, 1), 0x1000 * (k + 1)) for k in range(7)]
    root = leaves[0]
    for x in leaves[1:]:
        root = F.BinaryOpNode("max_op" if out != np.bool_ else "bit_or_op", root, x, (9, 8), out)
    src = F.generate_source(F._Program(root), kinds, 1, np.dtype(out), True, "flat")
    assert rtc_build(src, F.RTC_OPTIONS)[:4] == b"\x7fELF"


def _same(got, want):
    assert got.dtype == want.dtype and got.shape == want.shape
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("cols", [1, 2, 3, 4, 5, 8, 50, 63, 255, 257, 1000, 1001, 4097])
def test_flat_matches_numpy(cols, native):
    """Row vectors, one value per row, padded and odd rows, transposed and
    reversed leaves; few rows (row launch), and outputs that end inside, at
    and past a tile (flat launch)."""
    g = np.random.default_rng(cols)
    cp.set_config(native_dispatch=native)
    try:
        for rows in (1, 5, 65535 // cols + 1, 69632 // cols + 1, 90000 // cols + 3):
            x = g.standard_normal((rows, cols), dtype=np.float32)
            wide = g.standard_normal((rows, cols + 4), dtype=np.float32)
            r, c = g.standard_normal(cols, dtype=np.float32), g.standard_normal((rows, 1),
                                                                                dtype=np.float32)
            t = g.standard_normal((cols, rows), dtype=np.float32)
            i = g.integers(-9, 9, (rows, cols)).astype(np.int32)
            dx, dwide, dr, dc, dt, di = (cp.array(a) for a in (x, wide, r, c, t, i))
            _same(((dx - dr) / dr).get(), (x - r) / r)
            _same(((dx - dc) * dr).get(), (x - c) * r)
            _same((dx * dwide[:, :cols] - dr).get(), x * wide[:, :cols] - r)
            _same((dx * dwide[:, 3:3 + cols] - dc).get(), x * wide[:, 3:3 + cols] - c)
            _same((dx + dt.T - dr).get(), x + t.T - r)
            _same((dx[:, ::-1] * dr + dc).get(), x[:, ::-1] * r + c)
            _same((dr + dc).get(), r + c)
            _same((di * di[:1] + dc).get(), i * i[:1] + c)
            _same((dx > dr).get(), x > r)
            _same(cp.where(di > di[:, :1], dx, dr).get(), np.where(i > i[:, :1], x, r))
    finally:
        cp.set_config(native_dispatch=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float16, np.float64, np.int16, np.int64, np.bool_])
def test_flat_element_types(dtype):
    g = np.random.default_rng(5)
    for rows, cols in itertools.product((3, 20001), (6, 33, 48)):
        x, r, c = ((g.integers(0, 2, s) if dtype == np.bool_ else g.integers(-50, 50, s)).astype(dtype)
                   for s in ((rows, cols), (cols,), (rows, 1)))
        dx, dr, dc = cp.array(x), cp.array(r), cp.array(c)
        _same(cp.maximum(cp.maximum(dx, dr), dc).get() if dtype != np.bool_ else ((dx | dr) & dc).get(),
              np.maximum(np.maximum(x, r), c) if dtype != np.bool_ else (x | r) & c)
        _same((dx == dr).get(), x == r)


@pytest.mark.parametrize("dtype", [np.float32, np.float16, np.float64])
def test_column_sum_source_compiles(dtype):
    leaves = [_leaf((9, 8), dtype, (8, 1), 0x1000 * (k + 1)) for k in range(3)]
    root = F.BinaryOpNode("mul_op", F.BinaryOpNode("sub_op", leaves[0], leaves[1], (9, 8), dtype),
                          leaves[2], (9, 8), dtype)
    src = F.generate_source(F._Program(root), ["v", "p", "r"], 1, np.dtype(dtype), False, "colsum")
    assert rtc_build(src, F.RTC_OPTIONS)[:4] == b"\x7fELF"


def test_column_sum_leaf_classes():
    """A class stands for the strides it is read with; others are refused."""
    for st, want in (((8, 1), "v"), ((13, 1), "v"), ((-8, 1), "v"), ((0, 1), "p"), ((3, 0), "r"),
                     ((0, 0), "r"), ((1, 9), None), ((16, 2), None), ((8, -1), None)):
        assert F._col_kinds([9], 8, [(8, 1), st]) == (want and ["v", want])
    assert F._col_kinds([9], 3, [(3, 1)]) is None and F._col_kinds([], 8, [(1,)]) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.float16])
@pytest.mark.parametrize("rows,cols", [(1_200_000, 4), (700_000, 7), (90_000, 50), (20_000, 255),
                                       (20_000, 257), (5000, 1001), (40, 110_000)])
def test_column_sums_of_expressions(rows, cols, dtype, monkeypatch):
    """sum / mean / var / std of lazy expressions down the columns, with row
    vectors, one value per row, padded and transposed leaves: NumPy's values
    of the same expression, accumulated in float64."""
    monkeypatch.setattr(F, "COL_SUM_MIN", 1 << 22)  # smaller than calls are sent there
    g = np.random.default_rng(cols)
    wide = (g.integers(-8, 9, (rows, cols + 3)) / 4).astype(dtype)
    x, r, c = wide[:, 1:cols + 1], (g.integers(1, 5, cols) / 2).astype(dtype), \
        g.integers(-3, 4, (rows, 1)).astype(dtype)
    dw, dr, dc = cp.array(wide), cp.array(r), cp.array(c)
    dx = dw[:, 1:cols + 1]
    def down(expr):  # the one-pass sum itself
        from macmetalpy_amd.ndarray import ndarray
        res = ndarray._empty_device((cols,), expr._dtype)
        assert F.run_col_sum(expr._fusion_node, expr._dtype, res._ptr, 1.0)
        return res

    for got, e in ((down((dx - dr) * dc), (x - r) * c), (down(dx * dx.copy() + dc), x * x + c)):
        want = np.sum(e.astype(np.float64), axis=0).astype(dtype)
        assert got.dtype == want.dtype and np.array_equal(got.get(), want, equal_nan=True)
    for got, e in ((cp.sum((dx - dr) * dc, axis=0), (x - r) * c),
                   (cp.sum(dx * dx.copy() + dc, axis=0, keepdims=True), x * x + c)):
        want = np.sum(e.astype(np.float64), axis=0, keepdims=got.ndim == 2).astype(dtype)
        assert got.dtype == want.dtype and np.array_equal(got.get(), want, equal_nan=True)
    got, e = cp.mean(dx * dr, axis=0), (x * r).astype(np.float64)
    want = e.mean(axis=0)
    tol = 2 * np.finfo(dtype).eps * np.abs(e).mean(axis=0) + np.finfo(dtype).tiny
    assert got.dtype == dtype and np.all(np.abs(got.get().astype(np.float64) - want) <= tol)
    if dtype != np.float16:
        v = x.astype(np.float64)
        assert np.allclose(cp.std(dx, axis=0).get(), v.std(axis=0), rtol=8 * np.finfo(dtype).eps)


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_callers_expression_is_evaluated_once(native, monkeypatch):
    """A lazy expression that its program holds is evaluated by the first
    reduction down its columns and kept for the next; var's own deviations,
    which nothing else holds, are not written at all."""
    monkeypatch.setattr(F, "COL_SUM_MIN", 1 << 18)
    ran = []
    monkeypatch.setattr(F, "run_col_sum", lambda *a, f=F.run_col_sum: ran.append(1) or f(*a))
    cp.set_config(native_dispatch=native)
    x = np.random.default_rng(2).integers(-8, 9, (6000, 50)).astype(np.float32)
    d = cp.array(x)
    for f, want in ((cp.sum, x * 2 + 1), (cp.mean, None), (cp.var, None), (cp.std, None)):
        t = d * 2.0 + 1.0
        first = f(t, axis=0).get()
        assert t._fusion_node is None
        if want is not None:
            assert np.array_equal(first, want.sum(axis=0)) and np.array_equal(t.get(), want)
    assert len(ran) == 2  # var and std
    assert np.allclose(cp.var(d, axis=0).get(), x.astype(np.float64).var(axis=0), rtol=1e-6)
    assert np.allclose(cp.var(d.T, axis=0).get(), x.T.astype(np.float64).var(axis=0), rtol=1e-6)
    assert len(ran) == 3  # not down the columns of a transposed view


@pytest.mark.parametrize("kinds,cols,n,wide,flat", [
    # rows that fill the row launch's workgroups, in the caches
    ("fp", 511, 12_000_000, 4, True), ("fp", 1023, 12_000_000, 4, False),
    ("fp", 3001, 12_000_000, 4, False), ("pr", 1023, 12_000_000, 4, False),
    ("fr", 1023, 12_000_000, 4, True), ("fr", 3001, 12_000_000, 4, False),
    ("fp", 4097, 12_000_000, 4, True), ("fp", 40_001, 12_000_000, 4, False),
    ("fq", 900, 12_000_000, 4, True), ("fq", 3500, 12_000_000, 4, False),
    ("fp", 1023, 12_000_000, 2, True), ("fp", 3001, 12_000_000, 2, False),
    ("fr", 3001, 12_000_000, 2, True), ("fq", 3500, 12_000_000, 2, True),
    ("fp", 130, 12_000_000, 8, True), ("fp", 255, 12_000_000, 8, False),
    ("fq", 300, 12_000_000, 8, False), ("fqv", 300, 12_000_000, 8, True),
    ("pr", 40_001, 12_000_000, 8, False),
    # larger than those
    ("fp", 3001, 70_000_000, 4, True), ("fp", 40_001, 70_000_000, 4, True),
    ("pr", 3001, 70_000_000, 4, False), ("qw", 3500, 70_000_000, 4, True),
    ("fp", 3001, 70_000_000, 2, True), ("pr", 3001, 70_000_000, 2, False),
    ("fq", 300, 70_000_000, 8, True), ("fp", 511, 70_000_000, 8, False),
    ("fp", 5001, 70_000_000, 8, True), ("pr", 5001, 70_000_000, 8, False),
    # 153 MB read, 38 written (a comparison's result): the caches hold it
    ("fp", 145_921, 19_000_000, 4, False)])
def test_rows_go_flat_where_that_was_quicker(kinds, cols, n, wide, flat):
    traffic = n * wide * (1 + sum(k in "fv" for k in kinds))
    assert F._flat_cols(list(kinds), cols, traffic, wide, False, 4096) is flat


_UNARY = ["sin", "cos", "tanh", "exp", "log1p", "sqrt", "arctan", "cbrt"]


@pytest.mark.gpu
@pytest.mark.parametrize("i,dtype,cols,rows", [(0, np.float64, 130, 3000), (1, np.float64, 200, 3000),
                                               (2, np.float32, 513, 700), (3, np.float32, 3001, 90),
                                               (4, np.float32, 4097, 40), (5, np.float32, 2052, 70),
                                               (6, np.float16, 1025, 300), (7, np.float64, 301, 60_000)])
def test_both_dispatchers_take_the_same_launch(i, dtype, cols, rows, monkeypatch):
    """The native rule and the Python one agree: the modes of the kernels that
    they ask for, for expressions that nothing else builds."""
    x, r, c = (cp.array(np.ones(s, dtype)) for s in ((rows, cols), (cols,), (rows, 1)))
    modes, source = [], F.generate_source
    monkeypatch.setattr(F, "generate_source", lambda *a, **k: modes.append(a[5]) or source(*a, **k))
    for native in (True, False):
        cp.set_config(native_dispatch=native)
        y = getattr(cp, _UNARY[i])(cp.fmax(cp.fmin(x - r, x * c), r - c))
        (cp.floor(y) if native else cp.ceil(y))._materialize_if_lazy()
    assert len(modes) == 2 and modes[0] == modes[1]
