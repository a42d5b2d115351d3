"""Bounce-back nodes, whose populations a step leaves where they are, and lattices without cells, whose force fields are
not read, against the FP64 oracle: whole populations (solid interiors with a flow in them, beside closed faces), then
cells added to the flow."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu


def _mask(kind, shape):
    m = np.zeros(shape, dtype=np.uint8)
    if kind == "block":  # a solid block inside, walls two nodes thick beside it
        m[3:9, 4:11, 2:8] = 1
        m[:, :2, :] = m[:, -2:, :] = 1
    elif kind == "random":
        m[np.random.default_rng(3).random(shape) < 0.5] = 1
    elif kind == "solid":
        m[:] = 1
    else:  # velocity planes with a solid block between them
        m[:, :, 0], m[:, :, -1] = 2 + 4, 2 + 5
        m[4:9, 5:10, 4:9] = 1
    return m


@pytest.mark.parametrize("kind,periodic", [("block", (1, 1, 1)), ("block", (1, 0, 1)), ("block", (0, 0, 0)),
                                           ("random", (1, 0, 0)), ("random", (1, 1, 1)), ("solid", (0, 1, 1)),
                                           ("planes", (1, 1, 0))])
@pytest.mark.parametrize("precision", [0, 1])
def test_populations(kind, periodic, precision):
    import hemocell_amd as hc
    assert hc.NODE_BOUNCEBACK == 1 and hc.NODE_VELOCITY == 2
    shape = (13, 15, 17)
    mask = _mask(kind, shape)
    u = cases.units()
    g = hc.Simulation(0)
    g.lattice_init(*shape, u.tau, periodic=periodic, node_type=mask, precision=precision)
    o = OracleSim(*shape, u.tau, periodic=periodic, node_type=mask)
    f0 = None
    for s in (g, o):
        s.init_equilibrium(1.0, [1e-2, 5e-3, -2e-3])
        s.set_body_force([1e-5, 0, 2e-5])
        if kind == "planes":
            s.set_wall_velocity(4, [1e-2, 0, 0])
            s.set_wall_velocity(5, [-1e-2, 0, 0])
    for n in (1, 2, 3, 1):
        for s in (g, o):
            s.step(n)
        fg, fo = g.populations(), o.populations()
        assert np.abs(fg - fo).max() <= (1e-13 if precision == 0 else 2e-6)
    g.close()


def test_cells_added_to_a_flow():
    import hemocell_amd as hc
    u = cases.units()
    shape = (24, 30, 24)
    mask = np.zeros(shape, dtype=np.uint8)
    mask[:, :3, :] = mask[:, -3:, :] = 1  # a fifth of the nodes: the velocity pass leaves them out
    sims = []
    for cls in (0, 1):
        s = hc.Simulation(0) if cls == 0 else OracleSim(*shape, u.tau, periodic=(1, 1, 1), node_type=mask)
        if cls == 0:
            s.lattice_init(*shape, u.tau, periodic=(1, 1, 1), node_type=mask)
        s.init_equilibrium(1.0, [0, 0, 0])
        s.set_body_force([0, 0, 1e-5])
        s.set_force_limit(u.f_limit)
        s.step(5)
        model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
        x = cases.place(v * (1.02, 0.99, 0.99), (12, 15, 12))
        s.add_cells(s.add_cell_type(model, v, t, p, inner), x[None])
        s.step(6)
        sims.append(s)
    (xa, va, fa), (xo, vo, fo) = (s.vertices() for s in sims)
    assert cases.rel_l2(xa, xo) < 1e-12
    assert cases.rel_l2(va, vo) < 1e-9
    assert cases.rel_l2(fa, fo) < 1e-9
    assert np.abs(sims[0].populations() - sims[1].populations()).max() <= 1e-12
    sims[0].close()
