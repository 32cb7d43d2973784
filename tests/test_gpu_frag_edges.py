"""Fragments at the edges of what a thread of the fragment kernel holds (10
vertices in FP64, 12 in FP32), against the workgroup-per-cell kernel: cells of 6
to 14 edges whose corners one large triangle cuts one by one, and triangles
inside a cell; masses, value, Hessian, moments of both orders, adjoint and
fragment polygons."""
import numpy as np
import pytest

from mongeampere_amd import configs

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the same sums in another order


def _problem(edges, big):
    t = 2 * np.pi * (np.arange(edges) + 0.31) / edges
    X = np.concatenate([[[0.5, 0.5]], 0.5 + 0.3 * np.stack([np.cos(t), np.sin(t)], 1)])
    if big:  # one triangle whose edges cut corners of the central cell, and its surroundings
        s = 2 * np.pi * (np.arange(3) + 0.1) / 3
        vxy = np.concatenate([0.5 + 0.3 * np.stack([np.cos(s), np.sin(s)], 1),
                              0.5 + 2.0 * np.stack([np.cos(s), np.sin(s)], 1)])
        tri = [[0, 1, 2]] + [q for i in range(3) for q in ([i, i + 3, (i + 1) % 3 + 3],
                                                          [i, (i + 1) % 3 + 3, (i + 1) % 3])]
        tri = np.array(tri, np.int32)
    else:
        vxy, tri = configs.grid_mesh(40)
    return configs.Mesh(vxy, 1.0 + 0.3 * vxy[:, 0] + 0.2 * vxy[:, 1] ** 2, tri), X


@pytest.mark.parametrize("big", [True, False])
@pytest.mark.parametrize("edges", [6, 8, 9, 10, 11, 12, 13, 14])
def test_against_workgroup_kernel(engine, edges, big):
    mesh, X = _problem(edges, big)
    w = np.zeros(len(X))
    engine.set_mesh(mesh).set_diracs(X)

    def everything():
        f, g, H = engine.kantorovich(w)
        m, mom, second = engine.second_moment(w)
        dY, dval = engine.adjoint(w)
        cell, tri, start, xy = engine.fragments(w)
        return [np.array([f]), g, H.toarray(), m, mom, second, dY, dval], (cell, tri, start)

    a, fa = everything()
    _, g32, H32 = engine.kantorovich(w, "mixed")
    engine.set_option("force_general", 2)
    try:
        b, fb = everything()
    finally:
        engine.set_option("force_general", 0)
    for x, y in zip(a, b):
        assert np.abs(x - y).max() <= TOL * np.abs(y).max()
    for x, y in zip(fa, fb):
        assert np.array_equal(x, y)
    # FP32 geometry: masses within 2e-5 of the mean mass, Hessian within 1e-4
    assert np.abs(g32 - b[1]).max() <= 2e-5 * b[1].mean()
    assert np.abs(H32.toarray() - b[2]).max() <= 1e-4 * np.abs(b[2]).max()
