"""Steps with repulsion, where the cell kernel leaves the next spread to its own pass, against the separate kernels
and the FP64 oracle: several mechanics and velocity timescales, forces beyond the limit, extra forces, wall repulsion."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mech,vel,wall,limit,extra", [(1, 1, 0, 1.0, 0), (2, 1, 0, 1e-6, 1), (1, 3, 1, 1.0, 1),
                                                       (3, 2, 1, 1e-6, 0)])
def test_steps_agree(monkeypatch, mech, vel, wall, limit, extra):
    import hemocell_amd as hc
    u = cases.units()
    shape = (24, 22, 26)
    kw = dict(periodic=(1, 0, 1), node_type=cases.channel_mask(*shape, axis=1)) if wall else dict(periodic=(1, 1, 1))
    plt = [(12, 11, 10.5), (1, 2.2, 24), (2, 18.8, 25)] if wall else [(12, 11, 10.5), (1, 21, 24), (2, 0.5, 25)]
    sims = []
    for fuse in ("1", "0", "oracle"):
        monkeypatch.setenv("HC_FUSE", fuse if fuse != "oracle" else "1")
        s = OracleSim(*shape, u.tau, **kw) if fuse == "oracle" else hc.Simulation(0)
        if fuse != "oracle":
            s.lattice_init(*shape, u.tau, **kw)
        s.init_equilibrium(1.0, [0, 0, 1e-3])
        rng = np.random.default_rng(7)
        for kind, at in (("RBC", [(12, 11, 8), (12, 11, 13)]), ("PLT", plt)):
            model, v, t, p, inner = cases.mesh(kind, u, hc.build_mesh)
            s.add_cells(s.add_cell_type(model, v, t, p, inner, mech),
                        np.stack([cases.place(v * (1.03, 0.98, 1.0), c, cases.rotation(rng)) for c in at]))
        s.set_force_limit(u.f_limit * limit)
        s.set_repulsion(2e-5, 0.9, 2)
        if wall:
            s.set_boundary_repulsion(2e-5, 1.9, 2)
        s.set_velocity_timescale(vel)
        if extra and fuse != "oracle":
            s.set_extra_vertex_force(np.array([3, 500], dtype=np.int64), np.array([[1e-4, 0, 0], [-1e-4, 0, 0]]))
        for n in (1, 4, 3):
            s.step(n)
        sims.append(s)
    (xa, va, fa), (xb, vb, fb), (xo, vo, fo) = (s.vertices() for s in sims)
    for x, v, f in ((xb, vb, fb),) if extra else ((xb, vb, fb), (xo, vo, fo)):
        assert cases.rel_l2(xa, x) < 1e-11
        assert cases.rel_l2(va, v) < 1e-9
        assert cases.rel_l2(fa, f) < 1e-8
    assert np.abs(sims[0].repulsion_force()).max() > 0
    assert cases.rel_l2(sims[0].repulsion_force(), sims[1].repulsion_force()) < 1e-9
    if wall:
        assert np.abs(sims[0].boundary_repulsion_force()).max() > 0
    for s in sims[:2]:
        s.close()
