"""Cell and fluid statistics: every mesh size class against numpy, more cells than the pinned slot holds, and the
statistics' scratch not disturbing the run."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def _sim(n=(48, 48, 48), precision=0):
    import hemocell_amd as hc
    u = cases.units()
    s = hc.Simulation(0)
    s.lattice_init(*n, u.tau, precision=precision)
    s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
    s.set_force_limit(u.f_limit)
    return s, u


# positions of up to 2700 vertices in LDS; 8738 cells in the pinned slot
@pytest.mark.parametrize("triangles,ncells", [(20, 3), (600, 5), (2000, 2), (8000, 1), (20, 8738), (20, 8739)])
def test_cell_statistics(triangles, ncells):
    import hemocell_amd as hc
    s, u = _sim()
    v, t = hc.build_mesh(0, 8.0, triangles)
    _, _, _, params, _ = cases.mesh("RBC", u, hc.build_mesh)
    rng = np.random.default_rng(triangles + ncells)
    x = np.einsum("vj,cjk->cvk", v, np.eye(3) + 0.1 * rng.normal(size=(ncells, 3, 3))) + rng.uniform(5, 40, (ncells, 1, 3))
    s.add_cells(s.add_cell_type(hc.MODEL_RBC, v, t, params), x)
    vel = rng.normal(size=x.shape)
    s.set_vertices(v=vel.reshape(-1, 3))
    got = s.cell_stats()
    for c in list(range(min(ncells, 4))) + [ncells - 1]:
        a, b, d = (x[c][t[:, k]] for k in range(3))
        cr = np.cross(b - a, d - a)
        assert np.isclose(got["area"][c], 0.5 * np.linalg.norm(cr, axis=1).sum(), rtol=1e-12)
        p = x[c] - x[c][0]
        vol = (p[t[:, 0]] * np.cross(p[t[:, 1]], p[t[:, 2]])).sum() / 6.0
        assert np.isclose(got["volume"][c], vol, rtol=1e-11)
        assert np.allclose(got["centroid"][c], x[c].mean(0), rtol=1e-12)
        assert np.allclose(got["velocity"][c], vel[c].mean(0), atol=1e-14)
        assert np.array_equal(got["bbox"][c], np.stack([x[c].min(0), x[c].max(0)], -1).ravel())
        far = max(np.sqrt(((x[c] - q) ** 2).sum(1)).max() for q in x[c])
        assert np.isclose(got["stretch"][c], far, rtol=1e-15)
    s.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_statistics_between_steps_change_nothing(precision):
    import hemocell_amd as hc
    runs = []
    for look in (False, True):
        s, u = _sim((33, 31, 35), precision)
        model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
        s.add_cells(s.add_cell_type(model, v, t, p, inner), cases.place(v * (1.02, 0.99, 0.99), (16, 15, 17))[None])
        for _ in range(4):
            s.step(3)
            if look:
                f = s.fluid_stats("force")
                w = s.fluid_stats("velocity")
                _, uu = s.fluid()
                m = np.linalg.norm(uu, axis=1)
                assert np.isclose(w["max"], m.max(), rtol=1e-6) and np.isclose(w["avg"], m.mean(), rtol=1e-6)
                assert f["ncells"] == s.N and f["max"] > 0
        runs.append(s.vertices())
        s.close()
    for a, b in zip(*runs):
        assert cases.rel_l2(b, a) < (1e-6 if precision else 1e-12)
