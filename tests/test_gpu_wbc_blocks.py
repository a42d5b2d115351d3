"""White cells' FP32 forces over the ring-ordered and the compact tables against the padded lists and the FP64 oracle,
where the number of threads asked for is the one that runs (as many cells as compute units) and at the largest mesh whose
float offsets are staged; larger ones keep doubles and never read these tables."""
import numpy as np
import pytest

import cases
import geodesic
from oracle import OracleSim

pytestmark = pytest.mark.gpu


# 162 vertices fill a part of 256 threads, 642 all of 512 and part of 1024; 4002: staged up to about 4270
@pytest.mark.parametrize("frequency,ncells,block", [(4, 256, "256"), (4, 257, "512"), (8, 256, "512"), (8, 256, "1024"),
                                                    (20, 1, None)])
def test_forces(monkeypatch, frequency, ncells, block):
    import hemocell_amd as hc
    u = cases.units()
    v, t = geodesic.sphere(frequency, 8.0)
    params = cases.params(cases.WBC_MAT, len(t), u, 2)
    inner = np.array([(a, b) for a, b in enumerate(((v[:, None] + v[None, ::7]) ** 2).sum(2).argmin(1) * 7) if a < b],
                     dtype=np.int32)
    at = np.random.default_rng(frequency).uniform(0, 48, (ncells, 3))
    x = (v * (1.03, 0.98, 0.99))[None] + at[:, None]
    out = []
    for tables in ("csr", "compact", None, "oracle"):
        for name, value in (("HC_MECH_TABLES", tables), ("HC_WBC_BLOCK", block)):
            monkeypatch.setenv(name, value) if value and value != "oracle" else monkeypatch.delenv(name, raising=False)
        s = OracleSim(48, 48, 48, u.tau) if tables == "oracle" else hc.Simulation(0)
        if tables != "oracle":
            s.lattice_init(48, 48, 48, u.tau, precision=1)
        s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
        s.add_cells(s.add_cell_type(2, v, t, params, inner), x)
        s.step(1)  # in a uniform flow
        out.append(s.vertices()[2])
        if tables != "oracle":
            s.close()
    # offsets up to 16 lu with 24 bits over edges h strained by 2%, on forces that cancel around a vertex to h / 8 of an
    # edge's, twice that; 16 * 2^-24 / 0.02 of a force's other terms, a few of each kind
    h = 8 * 1.2 / frequency
    tol = max(3e-4, 2 * (2 * 16 * 2.0 ** -25 / (0.02 * h)) * (8 / h))
    for f in out[:3]:
        assert cases.rel_l2(f, out[3]) < tol
    assert cases.rel_l2(out[2], out[0]) < tol and cases.rel_l2(out[1], out[0]) < tol
