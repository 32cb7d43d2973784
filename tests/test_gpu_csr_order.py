"""ma_solve_laplacian_csr on rows whose columns come in any order, from the
size of a dense coarsest level (192) on: rows of up to 64 and of more entries
per aggregate, one to three coarse levels."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from mongeampere_amd.api import _ptr

pytestmark = pytest.mark.gpu


def _laplacian(n, per_row, rng):
    """A connected graph: the path 0..n-1 and per_row random edges a node."""
    i, j = np.repeat(np.arange(n), per_row), rng.integers(0, n, n * per_row)
    i, j = i[i != j], j[i != j]
    a, b = np.r_[i, np.arange(n - 1)], np.r_[j, np.arange(1, n)]
    w = rng.uniform(0.5, 2.0, len(a))
    H = sp.coo_matrix((-np.r_[w, w], (np.r_[a, b], np.r_[b, a])), shape=(n, n)).tocsr()
    return sp.csr_matrix(H - sp.diags(np.asarray(H.sum(axis=1)).ravel()))


def _solve(engine, ptr, col, val, g):
    n = len(ptr) - 1
    d, res, it = np.empty(n), ctypes.c_double(), ctypes.c_int64()
    engine._check(engine._L.ma_solve_laplacian_csr(
        engine._h, n, _ptr(ptr), _ptr(col), _ptr(val), _ptr(g), _ptr(d), 1e-12, 0,
        ctypes.byref(res), ctypes.byref(it)))
    return d, it.value


@pytest.mark.parametrize("n,per_row", [(192, 40), (193, 40), (196, 190), (400, 8), (400, 400),
                                       (1025, 60), (5000, 20)])
def test_any_order(engine, n, per_row):
    rng = np.random.default_rng(n + per_row)
    H = _laplacian(n, per_row, rng)
    H.sort_indices()
    ptr, col, val = H.indptr.astype(np.int32), H.indices.astype(np.int32), H.data.copy()
    g = rng.uniform(-1, 1, n)
    ref, ref_it = _solve(engine, ptr, col, val, g)
    mixed, mval = col.copy(), val.copy()
    for i in range(n):
        p = rng.permutation(ptr[i + 1] - ptr[i])
        mixed[ptr[i]:ptr[i + 1]] = col[ptr[i]:ptr[i + 1]][p]
        mval[ptr[i]:ptr[i + 1]] = val[ptr[i]:ptr[i + 1]][p]
    kept = mixed.copy(), mval.copy()
    d, it = _solve(engine, ptr, mixed, mval, g)
    # the same matrix, brought into the same order: the same bits
    assert np.array_equal(d, ref) and it == ref_it
    assert np.array_equal(mixed, kept[0]) and np.array_equal(mval, kept[1])
    A = H[:-1, :-1]
    assert d[-1] == 0.0
    # the stopping test, with the rounding of a product with A
    assert np.linalg.norm(A @ d[:-1] - g[:-1]) <= 2e-12 * np.linalg.norm(g[:-1]) + \
        1e-15 * np.linalg.norm(abs(A) @ np.abs(d[:-1]))
