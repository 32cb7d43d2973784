"""Copies between the caller's and the device's order, at counts around the
blocks of the prefix sum (1024 entries, counts of n + 1), with the work buffers
of a larger problem still in place: permuting the Diracs permutes every
output, in both layouts of the positions."""
import numpy as np
import pytest

from mongeampere_amd import configs

pytestmark = pytest.mark.gpu

# the outputs are the same sums in another order: a few hundred terms per
# cell, each with rounding 1.1e-16
TOL = 1e-13


def _mesh(n):
    vxy, tri = configs.grid_mesh(n, 0.0, 0.0, 1.0, 1.0)
    return configs.Mesh(vxy, 1.0 + vxy[:, 0] + 0.5 * vxy[:, 1], tri)


def _close(a, b):
    assert np.abs(a - b).max() <= TOL * max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("n", [1, 2, 1022, 1023, 1024, 1025, 5000])
def test_permuted_diracs(engine, n):
    rng = np.random.default_rng(n)
    mesh = _mesh(17)
    engine.set_mesh(mesh).set_diracs(rng.uniform(0.02, 0.98, (6000, 2)))
    engine.kantorovich(np.zeros(6000))
    X = rng.uniform(0.02, 0.98, (n, 2))
    w = rng.uniform(0.0, 0.1 / n, n)
    p = rng.permutation(n)
    out = []
    for Y, u in ((X, w), (X[p], w[p]), (np.asfortranarray(X), w)):
        engine.set_diracs(Y)
        m, mom, ine = engine.second_moment(u)
        m1, mom1 = engine.first_moment(u)
        _close(m1, m)
        _close(mom1, mom)
        f, g, H = engine.kantorovich(u)
        _close(g, m)
        if n > 1:  # (an empty cell, or a single one, shares no edge: its row is empty)
            assert np.all(np.diff(H.indptr)[g > 0] >= 1)
        for i in range(n):  # columns ascending in the caller's numbering
            assert np.all(np.diff(H.indices[H.indptr[i]:H.indptr[i + 1]]) > 0)
        out.append((m, mom, ine, H, f))
    (m, mom, ine, H, f), (mp, momp, inep, Hp, fp), (mf, momf, inef, Hf, ff) = out
    for a, b in ((mp, m[p]), (momp, mom[p]), (inep, ine[p]), (mf, m), (momf, mom), (inef, ine)):
        _close(a, b)
    for A, B in ((Hp, H[p][:, p]), (Hf, H)):
        scale = max(abs(B).max(), 1e-300) if B.nnz else 1.0
        assert abs(A - B).max() <= 1e-9 * scale  # edge lengths carry the vertices' rounding
    assert abs(fp - f) <= 1e-11 * max(abs(f), 1e-3) and abs(ff - f) <= 1e-11 * max(abs(f), 1e-3)
