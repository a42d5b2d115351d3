"""Platelet edges evaluated once each in LDS (meshes up to 227 vertices in FP64, 455 in FP32) against the kernels that
evaluate them by vertex: below, at and above those sizes, alone and with many cells, with forces beyond the
viscosity's limit."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,triangles,ncells,speed", [(0, 20, 3, 0.0), (0, 128, 400, 0.0), (0, 400, 2, 0.0),
                                                              (0, 600, 2, 0.0), (1, 128, 400, 0.0), (1, 800, 2, 0.0),
                                                              (1, 1200, 2, 0.0), (0, 128, 2, 30.0)])
def test_forces_by_edge(monkeypatch, precision, triangles, ncells, speed):
    import hemocell_amd as hc
    u = cases.units()
    v, t = hc.build_mesh(0, 4.0, triangles)
    _, _, _, params, _ = cases.mesh("PLT", u, hc.build_mesh)
    rng = np.random.default_rng(triangles + ncells)
    x = np.einsum("vj,cjk->cvk", v, np.eye(3) + 0.02 * rng.normal(size=(ncells, 3, 3))) + rng.uniform(8, 40, (ncells, 1, 3))
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("HC_FUSE", fuse)
        s = hc.Simulation(0)
        s.lattice_init(48, 48, 48, u.tau, precision=precision)
        s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
        s.add_cells(s.add_cell_type(hc.MODEL_PLT, v, t, params), x)
        s.set_velocity_timescale(1000)
        s.step(1)
        if speed:  # the velocities of the next steps' membrane viscosity
            s.set_vertices(v=speed * np.random.default_rng(1).normal(size=(ncells * len(v), 3)) * 1e-3)
        s.step(2)
        out.append(s.vertices())
        s.close()
    (xa, va, fa), (xb, vb, fb) = out
    assert np.abs(fb).max() > 0
    assert cases.rel_l2(xa, xb) < (1e-13 if precision == 0 else 1e-7)
    # FP32: offsets up to 8 lu in float, forces from differences of 0.01 of them
    assert cases.rel_l2(fa, fb) < (1e-11 if precision == 0 else 2e-4)
