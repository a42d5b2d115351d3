"""Cell-cell repulsion from the per-node runs of vertices: crowded nodes (runs ordered by insertion up to 16 vertices
and by heap sort above), lattices down to one node per axis, closed faces and vertices outside them.  Against the
FP64 oracle, which visits the same pairs in the same order."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,periodic,ncells,spread", [
    ((24, 24, 24), (1, 1, 1), 2, 0.2), ((24, 24, 24), (1, 1, 1), 15, 0.02), ((24, 24, 24), (1, 1, 1), 17, 0.02),
    ((24, 20, 22), (0, 1, 0), 40, 6.0), ((3, 3, 3), (1, 1, 1), 4, 1.0), ((2, 3, 4), (1, 1, 1), 3, 1.0),
    ((1, 5, 2), (1, 0, 1), 5, 1.0), ((4, 4, 4), (0, 0, 0), 5, 2.0), ((4, 5, 3), (1, 0, 1), 6, 3.0),
    ((5, 3, 4), (0, 1, 1), 6, 3.0)])
def test_repulsion_forces(shape, periodic, ncells, spread):
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh("PLT", u, hc.build_mesh)
    rng = np.random.default_rng(ncells)
    mid = 0.5 * (np.array(shape) - 1.0)
    x = np.stack([v - v.mean(axis=0) + mid + rng.uniform(-spread, spread, 3) for _ in range(ncells)])
    g = hc.Simulation(0)
    g.lattice_init(*shape, u.tau, periodic=periodic)
    o = OracleSim(*shape, u.tau, periodic=periodic)
    got = []
    for s in (g, o):
        s.init_equilibrium(1.0, [0, 0, 0])
        s.add_cells(s.add_cell_type(model, v, t, p, inner), x)
        s.set_repulsion(2e-3, 1.2, 1)
        for _ in range(2):  # the bins are empty again after a launch
            s.stage("repulsion")
        got.append(s.repulsion_force())
    assert np.abs(got[1]).max() > 0
    assert np.abs(got[0] - got[1]).max() <= 1e-13 * np.abs(got[1]).max()
    g.close()
