"""The forces of a large white cell beside red cells in the FP32 form are those of double-precision mechanics, whether
compute units are left over for it or not."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side_gpos", [None, "0"])
# the red cells have the more vertices in all; far fewer cells than compute units (256), one more than them
@pytest.mark.parametrize("nrbc", [40, 252])
def test_forces(monkeypatch, nrbc, side_gpos):
    import hemocell_amd as hc
    monkeypatch.setenv("HC_SIDE_GPOS", side_gpos) if side_gpos else monkeypatch.delenv("HC_SIDE_GPOS", raising=False)
    u = cases.units()
    out = []
    for s in (hc.Simulation(0), OracleSim(126, 126, 126, u.tau)):
        if isinstance(s, hc.Simulation):
            s.lattice_init(126, 126, 126, u.tau, precision=1)
        s.init_equilibrium(1.0, [0, 0, 0])
        centres = 18 * (np.stack(np.meshgrid(*[np.arange(7)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5)
        for kind, at in (("RBC", centres[:nrbc]), ("WBC2562", centres[-5:])):
            model, v, t, p, inner = cases.mesh(kind, u, hc.build_mesh)
            d = (v - v.mean(axis=0)) * (1.02, 0.99, 0.99)
            s.add_cells(s.add_cell_type(model, v, t, p, inner), np.stack([d + c for c in at]))
        # nothing moves: the fluid is at rest and no force was spread yet
        s.step(1)
        out.append(s.vertices()[2][-5 * len(v):])
    # positions up to 126 with 53 bits over relative changes of 1%, a few dozen terms a vertex: 126 * 2^-53 / 0.01 * 30
    assert cases.rel_l2(out[0], out[1]) < 5e-11
