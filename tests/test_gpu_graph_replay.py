"""Solves long enough to be replayed from a HIP graph (recorded after 32
batches: 256 iterations with the multigrid cycle, 1024 with Jacobi), against the
same launches one by one."""
import os
import re

import numpy as np
import pytest
import scipy.sparse as sp

from mongeampere_amd import configs

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53
with open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       "mongeampere_amd", "csrc", "engine.hip")) as f:
    GRAPH_FROM = int(re.search(r"int kGraphFrom = (\d+);", f.read()).group(1))


def _scattered(a, b, n):
    """Laplacian of a graph numbered at random: the aggregates, runs of
    consecutive unknowns, mean nothing, and the solve takes long."""
    rng = np.random.default_rng(n)
    p = rng.permutation(n)
    w = rng.uniform(0.5, 2.0, len(a))
    H = sp.coo_matrix((-np.r_[w, w], (p[np.r_[a, b]], p[np.r_[b, a]])), shape=(n, n)).tocsr()
    return sp.csr_matrix(H - sp.diags(np.asarray(H.sum(axis=1)).ravel())), rng.normal(size=n)


def _grid(m):
    k = np.arange(m * m).reshape(m, m)
    return _scattered(np.r_[k[:, :-1].ravel(), k[:-1].ravel()],
                      np.r_[k[:, 1:].ravel(), k[1:].ravel()], m * m)


def _path(n):
    return _scattered(np.arange(n - 1), np.arange(1, n), n)


@pytest.mark.parametrize("make,size,tol,sweeps",
                         [(_path, 1000, 1e-12, 1), (_path, 3000, 1e-12, 1), (_path, 3000, 1e-6, 1),
                          (_path, 3000, 1e-12, 2), (_grid, 150, 1e-12, 1), (_grid, 150, 1e-6, 1)])
def test_replay_is_eager(engine, make, size, tol, sweeps):
    """FP64 and FP32 hierarchies, both cycles; the same bits every time."""
    H, g = make(size)
    engine.set_option("amg_sweeps", sweeps)
    try:
        out = []
        for graphs in (1, 0, 1, 0, 1):
            engine.set_option("graphs", graphs)
            out.append(engine.solve_laplacian_matrix(H, g, rel_tol=tol))
        d, res, it = out[0]
        assert it > (GRAPH_FROM + 2) * 8  # two replays at least
        for e in out[1:]:
            assert np.array_equal(e[0], d) and e[1] == res and e[2] == it
        A, m = abs(H), H.shape[0] - 1
        drift = 8 * EPS * it * A.sum(axis=1).max() * np.linalg.norm(d)
        assert np.linalg.norm(H[:m, :m] @ d[:m] - g[:m]) <= tol * np.linalg.norm(g[:m]) + drift
    finally:
        engine.set_option("amg_sweeps", 1).set_option("graphs", 1)


@pytest.mark.parametrize("maxiter", [263, 264, 265, 272, 275])
def test_limits_about_a_replay(engine, maxiter):
    """A limit inside, at and past the first replayed batches: the residual
    reported is the eager one."""
    H, g = _path(3000)
    text = []
    try:
        for graphs in (1, 0):
            engine.set_option("graphs", graphs)
            with pytest.raises(Exception, match=f"after {maxiter} iterations") as x:
                engine.solve_laplacian_matrix(H, g, maxiter=maxiter)
            text.append(re.sub(r"0x\w+", "", str(x.value)))
    finally:
        engine.set_option("graphs", 1)
    assert text[0] == text[1]


def test_jacobi(engine):
    """One Newton step with the Jacobi preconditioner.  The evaluations' sums
    differ by rounding from run to run, so the solutions agree to the stopping
    test times the condition of the Laplacian (a few times N), not bit by bit."""
    n = 150_000
    p = configs.config1(N=n, n=64)
    out = []
    try:
        for graphs in (1, 0, 1):
            engine.set_option("graphs", graphs)
            engine.set_mesh(p.mesh).set_diracs(p.X)
            w, st = engine.ot_solve(p.nu, maxiter=0, cg_tol=1e-12, preconditioner="jacobi",
                                    raise_on_error=False)
            assert st.cg_iter > (GRAPH_FROM + 2) * 32
            out.append(w)
    finally:
        engine.set_option("graphs", 1)
    for w in out[1:]:
        assert np.abs(w - out[0]).max() <= 10 * n * 1e-12 * np.abs(out[0]).max()
