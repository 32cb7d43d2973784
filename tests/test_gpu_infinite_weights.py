"""Weights without bounds: a Dirac of weight -inf (or the lowest double) owns
nothing and leaves the others as if it were not there; one of weight +inf owns
everything.  Through the ring search and the pyramid walk, with every cell built
from the per-bin owners (no rings, no walk), and by the general kernels."""
import numpy as np
import pytest

import oracle
from mongeampere_amd import configs

pytestmark = pytest.mark.gpu

TOL = 1e-10   # FP64: relative to the largest entry
MIXED = 2e-5  # mixed mode: masses, of the mean mass
LOWEST = -np.finfo(np.float64).max
OPTIONS = [dict(), dict(local_rings=0, walk_budget=0), dict(force_general=1),
           dict(force_general=2)]
DEFAULTS = dict(local_rings=8, walk_budget=1024, force_general=0)


def _mesh():
    vxy, tri = configs.grid_mesh(21)
    return configs.Mesh(vxy, 1.0 + vxy[:, 0] + 0.5 * vxy[:, 1], tri)


def _inputs(n):
    rng = np.random.default_rng(n)
    return rng.uniform(0, 1, (n, 2)), rng.uniform(-1, 1, n) * 0.1 / n


@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("low", [-np.inf, LOWEST])
@pytest.mark.parametrize("n,hidden", [(24, 1), (96, 1), (400, 3), (5000, 1), (5000, 60)])
def test_hidden(engine, n, hidden, low, options):
    """24 to 5000 Diracs: pyramids of 2 to 6 levels; 1 to 60 of them hidden."""
    mesh, (X, w) = _mesh(), _inputs(n)
    gone = np.sort(np.random.default_rng(hidden).permutation(n)[:hidden])
    keep = np.setdiff1d(np.arange(n), gone)
    _, og, oH = oracle.kantorovich(mesh, X[keep], w[keep])
    om, omom = oracle.first_moment(mesh, X[keep], w[keep])
    wh = w.copy()
    wh[gone] = low
    try:
        for k, v in options.items():
            engine.set_option(k, v)
        engine.set_mesh(mesh).set_diracs(X)
        for _ in range(2):  # from cold and from the last owners
            _, g, H = engine.kantorovich(wh)
            assert (g[gone] == 0.0).all()
            assert np.abs(g[keep] - og).max() <= TOL * og.max()
            assert H[gone].nnz == 0
            assert abs(H[keep][:, keep] - oH).max() <= TOL * abs(oH).max()
        _, g32, _ = engine.kantorovich(wh, "mixed")
        assert (g32[gone] == 0.0).all()
        assert np.abs(g32[keep] - og).max() <= MIXED * og.mean()
        m, mom = engine.first_moment(wh)
        assert np.abs(m[keep] - om).max() <= TOL * om.max()
        assert np.abs(mom[keep] - omom).max() <= TOL * np.abs(omom).max()
        # finite weights again: the owners kept from before are no trap
        _, og, _ = oracle.kantorovich(mesh, X, w)
        _, g, _ = engine.kantorovich(w)
        assert np.abs(g - og).max() <= TOL * og.max()
    finally:
        for k, v in DEFAULTS.items():
            engine.set_option(k, v)


@pytest.mark.parametrize("options", OPTIONS)
@pytest.mark.parametrize("n", [24, 400, 5000])
def test_owner_of_everything(engine, n, options):
    mesh, (X, w) = _mesh(), _inputs(n)
    w[n // 3] = np.inf
    expect = np.zeros(n)
    expect[n // 3] = 1.75  # the mass of the mesh
    try:
        for k, v in options.items():
            engine.set_option(k, v)
        engine.set_mesh(mesh).set_diracs(X)
        for precision in ("fp64", "fp64", "mixed"):
            _, g, _ = engine.kantorovich(w, precision)
            assert np.abs(g - expect).max() <= (TOL if precision == "fp64" else MIXED) * 1.75
    finally:
        for k, v in DEFAULTS.items():
            engine.set_option(k, v)


@pytest.mark.parametrize("n", [24, 400])
def test_nobody(engine, n):
    """No weight above -inf: no differences of weights, so nothing to expect
    of the masses, but no bin has an owner to read."""
    mesh, (X, w) = _mesh(), _inputs(n)
    _, og, _ = oracle.kantorovich(mesh, X, w)
    engine.set_mesh(mesh).set_diracs(X)
    for _ in range(2):
        engine.kantorovich(np.full(n, -np.inf))
        _, g, _ = engine.kantorovich(w)
        assert np.abs(g - og).max() <= TOL * og.max()
