"""LU and the substitution at the edges of their panels (32, 16 and 8 columns
by the number of rows left), row moves and batches, against NumPy's solution
and the factors' own product."""
import numpy as np
import pytest

import macmetalpy_amd as cp
from macmetalpy_amd._backend import HipBackend
from macmetalpy_amd._dtypes import dtype_code

pytestmark = pytest.mark.gpu


def _factor(a):
    """(LU, 0-based pivots, info) of a (batch, n, n) host array."""
    d = cp.array(a)._ensure_gpu()
    b, n = a.shape[:2]
    piv, info = (cp.array(np.full(s, -7, np.int32))._ensure_gpu() for s in ((b, n), (b,)))
    HipBackend().lu(dtype_code(a.dtype), d._ptr, b, n, piv._ptr, info._ptr)
    return d.get(), piv.get(), info.get()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch,n", [(3, 1), (2, 2), (5, 31), (4, 32), (3, 33), (2, 63), (300, 64),
                                     (2, 65), (1, 200), (2, 257), (1, 512), (1, 513), (1, 1024),
                                     (1, 1030), (1, 2049)])
def test_factors_multiply_back(batch, n, dtype):
    """P A = L U row for row: |L| <= 1 (partial pivoting), and the product is
    within the factorization's backward error bound, n u |L| |U|."""
    g = np.random.default_rng(n)
    a = g.standard_normal((batch, n, n)).astype(dtype)
    lu, piv, info = _factor(a)
    assert np.all(info == 0)
    for b in range(min(batch, 3)):
        L = np.tril(lu[b].astype(np.float64), -1) + np.eye(n)
        U = np.triu(lu[b].astype(np.float64))
        assert np.abs(L).max() <= 1.0
        perm = np.arange(n)
        for k in range(n):
            p = piv[b, k]
            assert k <= p < n
            perm[[k, p]] = perm[[p, k]]
        bound = (n + 1) * np.finfo(dtype).eps * (np.abs(L) @ np.abs(U))
        assert np.all(np.abs(a[b].astype(np.float64)[perm] - L @ U) <= bound)


@pytest.mark.parametrize("n", [40, 100])
def test_every_row_moves(n):
    """A matrix whose pivots are the rows in reverse, in a cycle, and already
    in place: swaps that meet the same rows again and none at all."""
    for perm in (np.arange(n)[::-1], np.roll(np.arange(n), 1), np.arange(n)):
        a = np.zeros((1, n, n))
        a[0, perm, np.arange(n)] = np.arange(n, 0, -1)  # one nonzero a column
        lu, piv, info = _factor(a)
        assert info[0] == 0 and np.array_equal(lu[0], np.diag(np.arange(n, 0, -1.0)))


def test_zero_and_nan_columns():
    """info is the first exactly zero pivot; an all-NaN column keeps its row."""
    for n, z in ((20, 7), (70, 50), (300, 299), (300, 0)):
        a = np.random.default_rng(n).standard_normal((2, n, n))
        a[1, :, z] = 0.0
        assert list(_factor(a)[2]) == [0, z + 1]
        with pytest.raises(np.linalg.LinAlgError):
            cp.linalg.solve(cp.array(a[1]), cp.array(a[0][0]))
    a = np.random.default_rng(1).standard_normal((1, 40, 40))
    a[0, :, 0] = np.nan
    assert _factor(a)[1][0, 0] == 0


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch,n,nrhs", [(1, 1, 1), (3, 31, 2), (2, 32, 9), (40, 33, 1), (1, 64, 100),
                                          (1, 300, 1), (2, 500, 8), (1, 1000, 20), (1, 2048, 8),
                                          (1, 2100, 8),
                                          (1, 4200, 5)])
def test_solve(batch, n, nrhs, dtype):
    """Residual within the substitution's backward error: n u (|A| + |L| |U|)
    |x| is below 8 n u of |A| |x| for these diagonally weighted matrices."""
    g = np.random.default_rng(n + nrhs)
    a = g.standard_normal((batch, n, n)).astype(dtype) + (n ** 0.5 * np.eye(n)).astype(dtype)
    b = g.standard_normal((batch, n, nrhs)).astype(dtype)
    x = cp.linalg.solve(cp.array(a), cp.array(b)).get()
    assert x.dtype == dtype and x.shape == b.shape
    a, b, x = (t.astype(np.float64) for t in (a, b, x))
    bound = 8 * n * np.finfo(dtype).eps * (np.abs(a) @ np.abs(x) + np.abs(b))
    assert np.all(np.abs(a @ x - b) <= bound)


def _eliminate(a):
    """Elimination column by column with partial pivoting (the first row of
    largest |a|), each product and difference rounded by itself."""
    a, n, info = a.copy(), len(a), 0
    piv = np.arange(n)
    for k in range(n):
        p = k + int(np.argmax(np.abs(a[k:, k])))
        piv[k] = p
        a[[k, p]] = a[[p, k]]
        if a[k, k] == 0:
            info = info or k + 1
            continue
        a[k + 1:, k] /= a[k, k]
        a[k + 1:, k + 1:] -= a[k + 1:, k, None] * a[k, k + 1:]
    return a, piv, info


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batch,n", [(2, 31), (2, 33), (1, 65), (3, 100), (1, 129), (2, 200), (1, 255),
                                     (65, 260)])
def test_factors_are_elimination_by_columns(batch, n, dtype):
    """Below 256 unknowns, and for many matrices, blocks change nothing: the
    factors, pivots (with ties) and info are those of elimination column by
    column, bit for bit; repeated rows and columns of zeros are exactly singular."""
    g = np.random.default_rng(n)
    for kind in ("normal", "ties", "repeated row", "zero column", "wide range"):
        a = g.standard_normal((batch, n, n)).astype(dtype)
        if kind == "ties":
            a = np.sign(a) + (a > 1.5)
        if kind == "repeated row":
            a[:, n - 1] = a[:, 0]
        if kind == "zero column":
            a[:, :, n // 2] = 0
        if kind == "wide range":
            a *= (2.0 ** g.integers(-20, 20, a.shape)).astype(dtype)
        a = a.astype(dtype)
        lu, piv, info = _factor(a)
        for b in (0, batch - 1):
            want, wpiv, winfo = _eliminate(a[b])
            assert np.array_equal(piv[b], wpiv) and info[b] == winfo, kind
            assert np.array_equal(lu[b], want), kind
        if kind in ("repeated row", "zero column"):
            assert np.all(info > 0)
        if kind == "repeated row":
            with pytest.raises(np.linalg.LinAlgError):
                cp.linalg.solve(cp.array(a), cp.array(a[:, :, :1]))
