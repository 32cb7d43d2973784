"""The conjugate gradient's fused iteration at the edges of its kernels: levels
around the sizes at which the last ones become one workgroup's work (1024
rows, 192 for the dense solve), rows longer than the two entries a lane keeps,
both cycles, both precisions of the hierarchy, and Jacobi."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _laplacian(n, degree, seed):
    """A path plus random near neighbours, and a hub of 40 neighbours."""
    rng = np.random.default_rng(seed)
    a = np.concatenate([np.arange(n - 1)] + [rng.integers(0, n, n) for _ in range(degree)]
                       + [np.full(40, n // 2)])
    off = rng.integers(-9, 10, len(a))
    off[: n - 1] = 1
    off[-40:] = np.arange(-20, 20)
    b = np.clip(a + off, 0, n - 1)
    a, b = a[a != b], b[a != b]
    H = sp.coo_matrix((-rng.uniform(0.5, 2.0, len(a)), (a, b)), shape=(n, n)).tocsr()
    H = H + H.T
    return sp.csr_matrix(H - sp.diags(np.asarray(H.sum(axis=1)).ravel()))


def _check(H, g, d, res, it, tol):
    """The true residual: what the recurrence says, plus its drift (a few
    roundings of A x per iteration)."""
    m = H.shape[0] - 1
    assert d[-1] == 0.0 and res <= tol and it > 0
    r = np.linalg.norm(H[:m, :m] @ d[:m] - g[:m])
    drift = 8 * EPS * it * abs(H).sum(axis=1).max() * np.linalg.norm(d)
    assert r <= tol * np.linalg.norm(g[:m]) + drift


@pytest.mark.parametrize("n", [768, 769, 1024, 1025, 3073, 4096, 4097, 16385, 70001])
@pytest.mark.parametrize("sweeps", [1, 2])
def test_tail_of_the_cycle(engine, n, sweeps):
    H = _laplacian(n, 3, n)
    g = np.random.default_rng(n).normal(size=n)
    g -= g.mean()
    engine.set_option("amg_sweeps", sweeps)
    try:
        for tol in (1e-6, 1e-12):  # FP32 and FP64 hierarchy
            d, res, it = engine.solve_laplacian_matrix(H, g, rel_tol=tol)
            _check(H, g, d, res, it, tol)
    finally:
        engine.set_option("amg_sweeps", 1)


def test_one_iteration_and_limits(engine):
    """maxiter inside, at and past a batch of iterations: the count and the
    residual that are reported are those of the returned iterate."""
    n = 3000
    H = _laplacian(n, 3, 7)
    g = np.random.default_rng(7).normal(size=n)
    g -= g.mean()
    full = engine.solve_laplacian_matrix(H, g, rel_tol=1e-10)[2]
    assert full > 9
    m = n - 1
    for k in (1, 2, 7, 8, 9):
        with pytest.raises(Exception, match=f"after {k} iterations"):
            engine.solve_laplacian_matrix(H, g, rel_tol=1e-10, maxiter=k)
    d, res, it = engine.solve_laplacian_matrix(H, g, rel_tol=1e-10, maxiter=full)
    assert it == full
    r = np.linalg.norm(H[:m, :m] @ d[:m] - g[:m]) / np.linalg.norm(g[:m])
    assert abs(r - res) <= 1e-3 * res + 1e-12
    # a tolerance of 1 takes one iteration
    assert engine.solve_laplacian_matrix(H, g, rel_tol=1.0)[2] >= 1
