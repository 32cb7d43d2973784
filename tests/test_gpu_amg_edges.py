"""The multigrid set-up at the edges of its kernels, against a direct solve:
coarsest matrices around the register tiles of the dense inverse (64, 128 and
192 unknowns), one and several levels, and coarse rows of more entries than a
wave has lanes."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

pytestmark = pytest.mark.gpu


def _laplacian(n, degree, seed):
    """Symmetric weighted graph Laplacian: a path plus random near neighbours."""
    rng = np.random.default_rng(seed)
    i = np.arange(n - 1)
    a = [i] + [rng.integers(0, n, n) for _ in range(degree)]
    b = [i + 1] + [np.clip(x + rng.integers(-3 * degree, 3 * degree + 1, n), 0, n - 1) for x in a[1:]]
    a, b = np.concatenate(a), np.concatenate(b)
    a, b = a[a != b], b[a != b]
    w = rng.uniform(0.5, 2.0, len(a))
    H = sp.coo_matrix((-w, (a, b)), shape=(n, n)).tocsr()
    H = H + H.T
    return sp.csr_matrix(H - sp.diags(np.asarray(H.sum(axis=1)).ravel()))


@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 64, 65, 128, 129, 191, 192, 193, 767, 769, 3100])
@pytest.mark.parametrize("degree", [1, 3, 20])
def test_against_direct_solve(engine, n, degree):
    H = _laplacian(n, degree, n + degree)
    g = np.random.default_rng(n).normal(size=n)
    g -= g.mean()
    d, res, _ = engine.solve_laplacian_matrix(H, g)
    ref = np.append(spl.spsolve(sp.csc_matrix(H[:-1, :-1]), g[:-1]), 0.0)
    # the solve stops at a relative residual of 1e-12; a path of n unknowns
    # has a condition number of about n^2
    assert res <= 1e-12
    assert np.abs(d - ref).max() <= 1e-12 * max(n, 100) ** 2 * np.abs(ref).max()
