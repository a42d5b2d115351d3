"""FP64 mechanics from factors evaluated once per triangle and edge, against the evaluation by vertex
(HC_MECH_TABLES=csr): meshes from 12 to 2562 vertices, with and without membrane viscosity, and velocities beyond its
limit; the two orders of evaluation (all at once, or list after list where LDS is short) agree bit for bit."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,triangles,ncells,eta,speed", [
    ("RBC", 20, 3, 0.0, 0.0), ("RBC", 80, 2, 1.0, 1.0), ("RBC", 1280, 2, 0.0, 0.0), ("RBC", 1280, 300, 1.0, 1.0),
    ("RBC", 5000, 1, 0.0, 0.0), ("WBC", 1280, 2, 1.0, 1.0), ("WBC", 1280, 2, 1.0, 3e4), ("WBC", 5000, 1, 1.0, 1.0)])
def test_forces(monkeypatch, kind, triangles, ncells, eta, speed):
    import hemocell_amd as hc
    u = cases.units()
    v, t = hc.build_mesh(0, 7.0, triangles)
    model, v0, t0, params, inner = cases.mesh(kind, u, hc.build_mesh)
    params.eta_m = eta * (params.eta_m if params.eta_m else 1e-3)
    rng = np.random.default_rng(triangles + ncells)
    x = np.einsum("vj,cjk->cvk", v, np.eye(3) + 0.02 * rng.normal(size=(ncells, 3, 3))) + rng.uniform(12, 36, (ncells, 1, 3))
    vel = speed * 1e-3 * rng.normal(size=(ncells * len(v), 3))
    out = []
    for lds, tables in ((None, None), ("8192", None), (None, "csr")):
        for name, value in (("HC_SPREAD_LDS", lds), ("HC_MECH_TABLES", tables)):
            monkeypatch.setenv(name, value) if value else monkeypatch.delenv(name, raising=False)
        s = hc.Simulation(0)
        s.lattice_init(48, 48, 48, u.tau, precision=0)
        s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
        s.add_cells(s.add_cell_type(model, v, t, params), x)
        s.set_velocity_timescale(1000)
        s.step(1)
        s.set_vertices(v=vel, x=x.reshape(-1, 3))
        s.step(1)
        out.append(s.vertices())
        s.close()
    assert np.abs(out[0][2]).max() > 0
    assert np.array_equal(out[0][2], out[1][2])
    assert cases.rel_l2(out[0][0], out[2][0]) < 1e-14
    # forces from relative changes of 2% of areas and lengths, each to some 1e-15
    assert cases.rel_l2(out[0][2], out[2][2]) < 1e-11
