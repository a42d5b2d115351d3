"""The cell kernel's spread over marked support nodes, at the edges of its layout: boxes taller than one 64-node
mask word, one pass, many passes, and the vertex-by-vertex form when not even 64 sums fit; vertices on nodes, on
periodic faces and next to closed ones.  Against the FP64 oracle over three steps."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu


def _run(shape, periodic, xs, scale, precision, steps=3):
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
    v = v * scale
    g = hc.Simulation(0)
    g.lattice_init(*shape, u.tau, periodic=periodic, precision=precision)
    o = OracleSim(*shape, u.tau, periodic=periodic)
    for s in (g, o):
        s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
        s.set_force_limit(u.f_limit)
        s.add_cells(s.add_cell_type(model, v, t, p, inner), xs(v))
        s.step(steps)
    a, b = g.vertices(), o.vertices()
    x0 = xs(v).reshape(-1, 3)
    g.close()
    return cases.rel_l2(a[0] - x0, b[0] - x0), cases.rel_l2(a[1], b[1])


def _strained(v, centre, seed=0):
    rng = np.random.default_rng(seed)
    s = 0.02 * rng.uniform(-1, 1, (3, 3))
    d = v - v.mean(axis=0)
    return d + d @ (s + s.T) + np.asarray(centre)


# a 70-spacing cell: 3600 mask words (two per row); 8192 B cannot hold them, 45056 B leave 112 sums of ~5000,
# 98304 B ~1950
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("box", [None, 8192, 98304])
def test_tall_boxes(monkeypatch, box, precision):
    if box:
        monkeypatch.setenv("HC_SPREAD_LDS", str(box))
    dx, dv = _run((80, 32, 80), (1, 1, 1), lambda v: _strained(v, (40.3, 15.8, 39.6))[None], 4.5, precision)
    assert max(dx, dv) < (2e-5 if precision else 1e-10), (dx, dv)


# an ordinary cell: 8192 B hold ~200 of ~1290 sums, 21504 B ~680, the default all
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("box", [None, 8192, 21504])
@pytest.mark.parametrize("where", ["inside", "corner", "on_nodes", "closed"])
def test_passes_and_faces(monkeypatch, box, where, precision):
    if box:
        monkeypatch.setenv("HC_SPREAD_LDS", str(box))
    n, periodic = (31, 29, 33), (1, 1, 1)
    centre = {"inside": (15.2, 14.1, 16.7), "corner": (0.3, 28.9, -0.4), "on_nodes": (15.0, 14.0, 16.0),
              "closed": (9.0, 14.1, 16.7)}[where]
    if where == "closed":
        periodic = (0, 1, 0)

    def xs(v):
        x = _strained(v, centre)
        if where == "on_nodes":  # the mesh's vertices in the planes of symmetry lie on node planes
            x = (v - v.mean(axis=0)) * (1.02, 0.99, 0.99) + centre
            assert (np.abs(x - np.round(x)) < 1e-9).any(axis=1).sum() > 60
        if where == "closed":
            x[:, 0] += 0.4 - x[:, 0].min()  # supports end at the open face's last node
        return np.stack([x, x + (0.0, 0.0, 0.25)])
    dx, dv = _run(n, periodic, xs, 1.0, precision)
    assert max(dx, dv) < (2e-5 if precision else 1e-10), (dx, dv)
