"""Batches whose cells have several meshes, around the number of cells up to which they share one launch, against
every case stepped alone."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


# one launch holds the cells of every mesh up to the number of compute units (256 on this device), one launch per
# mesh more than that
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nplt", [3, 251, 252])
def test_meshes_sharing_a_launch(nplt, precision):
    import hemocell_amd as hc
    u = cases.units()
    rng = np.random.default_rng(nplt)

    def make(kind, centres):
        model, v, t, p, inner = cases.mesh(kind, u, hc.build_mesh)
        s = hc.Simulation(0)
        s.lattice_init(48, 48, 48, u.tau, precision=precision)
        s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
        s.set_force_limit(u.f_limit)
        d = (v - v.mean(axis=0)) * (1.02, 0.99, 0.99)
        s.add_cells(s.add_cell_type(model, v, t, p, inner), np.stack([d + c for c in centres]))
        return s
    where = [("RBC", [(20, 20, 20), (24, 20, 30)]), ("WBC", [(12, 30, 30), (30, 12, 12), (40, 40, 8)]),
             ("PLT", rng.uniform(0, 48, (nplt, 3)))]
    batch, alone = [make(*w) for w in where], [make(*w) for w in where]
    hc.step_batch(batch, 4)
    for a, b in zip(batch, alone):
        b.step(4)
        for p, q in zip(a.vertices()[:2], b.vertices()[:2]):
            assert cases.rel_l2(p, q) < (1e-5 if precision else 1e-12)
        a.close()
        b.close()
