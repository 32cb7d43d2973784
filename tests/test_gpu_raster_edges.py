"""Rasterisation at the edges of what a group of lanes covers, against the CPU
oracle: fragments of 1 to 16 and more pixels, of 512 and 513 (the next kernel's),
of more than 16 vertices, partly or wholly outside the image."""
import numpy as np
import pytest

import oracle
from mongeampere_amd import configs

pytestmark = pytest.mark.gpu

TOL = 1e-12  # of the largest pixel: a few hundred FP64 terms per pixel


def _draw(engine, mesh, X, w, box, W, H, nc=2):
    rng = np.random.default_rng(W * 1000 + H)
    colors = rng.uniform(size=(len(X), nc))
    engine.set_mesh(mesh).set_diracs(X)
    img = engine.draw_laguerre_diagram(w, colors, box, W, H)
    ref = oracle.draw_laguerre_diagram(mesh, X, w, colors, box, W, H)
    assert np.abs(img - ref).max() <= TOL * max(np.abs(ref).max(), 1e-300)


def _mesh(n):
    vxy, tri = configs.grid_mesh(n, 0.0, 0.0, 1.0, 1.0)
    return configs.Mesh(vxy, 1.0 + vxy[:, 0] + 0.5 * vxy[:, 1], tri)


@pytest.mark.parametrize("size", [(1, 1), (2, 3), (4, 4), (17, 1), (1, 17), (32, 16), (27, 19),
                                  (1, 512), (513, 1), (40, 40)])
@pytest.mark.parametrize("box", [(0.0, 0.0, 1.0, 1.0), (0.3, -0.4, 0.9, 0.7)])
def test_pixels_of_a_fragment(engine, size, box):
    # two triangles, one and three Diracs: fragments as large as the image
    _draw(engine, _mesh(2), np.array([[0.4, 0.3]]), np.zeros(1), box, *size)
    X = np.array([[0.3, 0.2], [0.7, 0.4], [0.5, 0.8]])
    _draw(engine, _mesh(2), X, np.zeros(3), box, *size)


@pytest.mark.parametrize("edges", [15, 16, 17, 20])
@pytest.mark.parametrize("size", [(9, 9), (64, 64)])
def test_vertices_of_a_fragment(engine, edges, size):
    t = 2 * np.pi * (np.arange(edges) + 0.25) / edges
    ring = np.c_[0.7 + 0.1 * np.cos(t), 0.25 + 0.1 * np.sin(t)]
    X = np.r_[[[0.7, 0.25]], ring]
    _draw(engine, _mesh(2), X, np.zeros(len(X)), (0.0, 0.0, 1.0, 1.0), *size)


def test_outside_the_image(engine):
    X = np.random.default_rng(3).uniform(0.05, 0.95, (200, 2))
    _draw(engine, _mesh(9), X, np.zeros(200), (0.9, 0.9, 1.7, 1.3), 20, 11)


@pytest.mark.parametrize("n", [1, 7, 31, 60, 300, 3000])
def test_fragment_slots(engine, n):
    """Slots reserved by whole workgroups: fragments from less than one wave
    to many workgroups, none lost or written twice."""
    X = np.random.default_rng(n).uniform(0.05, 0.95, (n, 2))
    mesh = _mesh(6)
    engine.set_mesh(mesh).set_diracs(X)
    cell, tri, start, xy = engine.fragments(np.zeros(n))
    assert len(set(zip(cell.tolist(), tri.tolist()))) == len(cell)  # one per pair
    assert start[0] == 0 and np.all(np.diff(start) >= 3) and start[-1] == len(xy)
    area = 0.0
    for a, b in zip(start[:-1], start[1:]):
        p = xy[a:b]
        q = np.roll(p, -1, axis=0)
        s = 0.5 * (p[:, 0] * q[:, 1] - p[:, 1] * q[:, 0]).sum()
        assert s > 0
        area += s
    assert abs(area - 1.0) <= 1e-12
