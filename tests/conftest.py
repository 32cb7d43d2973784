import json
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the C ABI on device 0)")
    config.addinivalue_line("markers", "slow: large inputs")


def load_golden(name):
    from mongeampere_amd.configs import Mesh

    with open(os.path.join(GOLDEN, f"{name}.json")) as f:
        d = json.load(f)
    mesh = Mesh(np.array(d["vxy"], np.float64), np.array(d["vval"], np.float64),
                np.array(d["tri"], np.int32))
    X = np.array(d["X"], np.float64)
    w = np.array(d["w"], np.float64)
    e = d["expected"]
    n = len(w)
    H = np.zeros((n, n))
    pattern = set()
    for i, j, v in e["hessian"]:
        H[i, j] += v
        pattern.add((i, j))
    return dict(name=name, mesh=mesh, X=X, w=w, fval=e["fval"], mass=np.array(e["mass"]),
                intg=np.array(e["intg"]), mom=np.array(e["mom"]), H=H, pattern=pattern,
                inertia=np.array(e["inertia"]), frags=np.array(e["fragments"]).reshape(-1, 5))


def frag_summary(cell, tri, start, xy):
    """{(Dirac, triangle): (area, centroid x, centroid y)} of a fragment list
    (vertices xy[start[f]:start[f+1]], counter-clockwise), by the shoelace
    formula about the first vertex."""
    out = {}
    for f in range(len(cell)):
        p = xy[start[f]:start[f + 1]]
        q = p - p[0]
        x0, y0 = q[1:-1, 0], q[1:-1, 1]
        x1, y1 = q[2:, 0], q[2:, 1]
        a = 0.5 * (x0 * y1 - x1 * y0)
        A = a.sum()
        cx = (a * (x0 + x1)).sum() / (3 * A) + p[0, 0]
        cy = (a * (y0 + y1)).sum() / (3 * A) + p[0, 1]
        key = (int(cell[f]), int(tri[f]))
        assert key not in out, f"fragment {key} listed twice"
        out[key] = (A, cx, cy)
    return out


GOLDEN_CASES = sorted(f[:-5] for f in os.listdir(GOLDEN) if f.endswith(".json"))


def w2_cells(engine, nu, w):
    """W2^2 at weights w near the optimum, as (per-cell terms, correction).

    The dual value -F(w) = sum_i [cost_i - w_i (m_i - nu_i)] (cost_i =
    int_{Lag_i} rho |x - y_i|^2) falls short of its maximum W2^2 by
    (1/2) g^T H^+ g + O(|g|^3), g = m - nu, H the Hessian at w (-F is concave
    with gradient -g and Hessian -H): the correction is the value of one
    Newton step, (1/2) g.d with H d = g (gauge-fixed solve).  A solve stopped
    at max relative error 1e-9 on 2e5 cells leaves ~1e-17 in -F(w), which a
    central difference with h = 1e-6 would turn into ~1e-6 of a gradient
    entry; the corrected value is exact to third order.  The per-cell terms
    let a difference of two values be summed cell by cell (math.fsum of the
    differences), keeping the precision of the cells instead of that of the
    totals."""
    _, m, _ = engine.kantorovich(w, precision="fp64", hessian=False)
    g = m - nu
    gc = g - g.mean()  # the total-mass rounding is no direction of descent
    d, _, _ = engine.solve_laplacian(gc, rel_tol=1e-10)
    return engine.cell_costs() - w * g, 0.5 * float(gc @ d)


def central_difference(plus, minus, h):
    """(W2^2(+h) - W2^2(-h)) / 2h from two w2_cells results."""
    import math

    (cp, kp), (cm, km) = plus, minus
    return (math.fsum((cp - cm).tolist()) + (kp - km)) / (2.0 * h)


@pytest.fixture(scope="session")
def engine():
    from mongeampere_amd.api import Engine

    e = Engine(0)
    yield e
    e.close()


def option_defaults():
    """{option: default} of Engine.set_option, from the engine's own header."""
    import re

    with open(os.path.join(ROOT, "mongeampere_amd", "csrc", "engine.h")) as f:
        text = f.read()
    constant = dict(re.findall(r"constexpr int (k\w+) = (\d+);", text))

    def default(member):
        v = re.search(r"\b%s = (?:ma::)?([\w.]+);" % member, text).group(1)
        return float(constant.get(v, v))

    return {"force_general": int(default("force_general")), "cap_cand": int(default("cap_cand")),
            "graphs": int(default("use_graphs")), "local_rings": int(default("local_rings")),
            "walk_budget": int(default("walk_budget")),
            "amg_omega_permille": round(1000 * default("amg_omega")),
            "amg_corr_permille": round(1000 * default("amg_corr")),
            "amg_sweeps": int(default("amg_sweeps")), "far_cells": int(default("far_cells"))}


def restore_options(engine):
    for name, value in option_defaults().items():
        engine.set_option(name, value)


@pytest.fixture(autouse=True)
def _default_options(request):
    """The engine is shared by the session: every test starts from the options
    a caller gets, whatever the test before it left."""
    if "engine" in request.fixturenames:
        restore_options(request.getfixturevalue("engine"))
    yield
