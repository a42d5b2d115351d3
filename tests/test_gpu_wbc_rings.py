"""White cells' FP32 forces over the ring-ordered and the compact tables, with inner links, against the padded lists and
the FP64 oracle: the meshes' smallest and largest sizes, one and several workgroup shapes."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("triangles,block", [(80, None), (600, "256"), (2000, "512"), (2000, None), (8000, None)])
def test_forces(monkeypatch, triangles, block):
    import hemocell_amd as hc
    u = cases.units()
    v, t = hc.build_mesh(0, 8.0, triangles)
    model, v0, t0, params, inner0 = cases.mesh("WBC", u, hc.build_mesh)
    n = len(v)
    # each vertex and its antipode, each pair once
    far = np.array([int(((v - q + 2 * (q - v.mean(0))) ** 2).sum(1).argmin()) for q in v])
    inner = np.array(sorted({(min(a, b), max(a, b)) for a, b in enumerate(far)}), dtype=np.int32)
    x = cases.place(v * (1.03, 0.98, 0.99), (20, 21, 20))[None]
    out = []
    for tables in ("csr", "compact", None, "oracle"):
        for name, value in (("HC_MECH_TABLES", tables), ("HC_WBC_BLOCK", block)):
            monkeypatch.setenv(name, value) if value and value != "oracle" else monkeypatch.delenv(name, raising=False)
        s = OracleSim(40, 42, 41, u.tau) if tables == "oracle" else hc.Simulation(0)
        if tables != "oracle":
            s.lattice_init(40, 42, 41, u.tau, precision=1)
        s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
        s.add_cells(s.add_cell_type(model, v, t, params, inner), x)
        s.step(2)
        out.append(s.vertices()[2])
        if tables != "oracle":
            s.close()
    # float offsets up to 16 lu and relative changes of 2%: 16 * 2^-24 / 0.02 of a force's terms, a few of each kind
    tol = 3e-4
    for f in out[:3]:
        assert cases.rel_l2(f, out[3]) < tol
    assert cases.rel_l2(out[2], out[0]) < tol and cases.rel_l2(out[1], out[0]) < tol
