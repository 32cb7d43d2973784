"""Newton solves whose tolerance lies about the representability floor of FP64
weights: a solve ends with MA_OK and an error within the tolerance, or stops
at the floor with an error above it; what it reports is what its weights give."""
import numpy as np
import pytest

from mongeampere_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [0.25, 0.5, 1.0, 2.0, 4.0])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tolerance_about_the_floor(engine, factor, precision):
    rng = np.random.default_rng(11)
    X = rng.uniform(0.05, 0.95, (1500, 2))
    X[:20] = X[20:40] + 2e-6 * rng.choice([-1.0, 1.0], (20, 2))
    vxy, tri = configs.grid_mesh(33, 0.0, 0.0, 1.0, 1.0)
    mesh = configs.Mesh(vxy, 1.0 + vxy[:, 0], tri)
    engine.set_mesh(mesh).set_diracs(X)
    w0 = np.full(1500, 0.25)  # ulp(w) = 5.6e-17
    _, m, H = engine.kantorovich(w0)
    nu = np.full(1500, m.sum() / 1500)
    off = abs(H - np.diag(H.diagonal())).max()
    tol = factor * off * 5.6e-17 / nu[0]
    for k in range(4):
        w, st = engine.ot_solve(nu, w0 + 1e-5 * k, stop="maxrel", tol=tol, precision=precision,
                                raise_on_error=False)
        _, g, _ = engine.kantorovich(w, hessian=False)
        err = np.abs(g - nu).max() / nu[0]
        assert abs(err - st.max_rel_err) <= 1e-12 + 1e-2 * err
        assert st.status in ("MA_OK", "MA_LINESEARCH_FAIL")
        assert (st.status == "MA_OK") == (st.max_rel_err <= tol)
