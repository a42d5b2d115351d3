"""State read back in chunks through pinned staging: what was set comes back bit for bit, for counts below,
across and just past the edges of a chunk (1 MB) and of a block."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def _sim(shape, precision, periodic=(1, 1, 1), mask=None):
    import hemocell_amd as hc
    s = hc.Simulation(0)
    s.lattice_init(*shape, 1.1, periodic=periodic, node_type=mask, precision=precision)
    s.init_equilibrium(1.0, (0, 0, 0))
    return s


# 1 MB holds 6898 nodes of 19 populations, 32768 of (rho, u), 43690 of u alone and 131072 of rho alone
@pytest.mark.parametrize("shape", [(3, 5, 7), (16, 16, 16), (6898, 1, 1), (6899, 1, 1), (32, 32, 32), (32769, 1, 1), (70, 61, 43)])
def test_populations_and_fluid(shape):
    rng = np.random.default_rng(3)
    N = int(np.prod(shape))
    s = _sim(shape, 0)
    f = 1e-2 * rng.uniform(-1, 1, size=(19, N))
    s.set_populations(f)
    assert np.array_equal(s.populations(), f)
    rho, u = s.fluid()
    rho1, none = s.fluid(velocity=False)
    assert none is None and np.array_equal(rho, rho1)
    assert np.allclose(rho, 1.0 + f.sum(0), rtol=1e-14, atol=1e-15)
    z = f[[7, 9, 12, 15, 17]].sum(0) - f[[3, 6, 8, 16, 18]].sum(0)
    assert np.allclose(u[:, 2], z / rho, rtol=1e-12, atol=1e-16)
    only = np.zeros((N, 3))
    import hemocell_amd as hc
    s._chk(s.lib.hc_get_fluid(s.h, None, hc._dp(only)))
    assert np.array_equal(only, u)
    s.close()


# 1 MB holds 14563 vertices of three fields, 21845 of two and 43690 of one; an RBC has 642
@pytest.mark.parametrize("ncells", [1, 22, 23, 34, 35, 68, 69, 140])
def test_vertices(ncells):
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
    rng = np.random.default_rng(ncells)
    s = _sim((64, 64, 64), 0)
    x = np.stack([cases.place(v, rng.uniform(20, 40, 3)) for _ in range(ncells)])
    s.add_cells(s.add_cell_type(model, v, t, p, inner), x)
    a = [rng.normal(size=(ncells * len(v), 3)) for _ in range(3)]
    s.set_vertices(*a)
    for got, want in zip(s.vertices(), a):
        assert np.array_equal(got, want)
    for pick in ((0, 1), (1, 2), (2,)):
        out = [np.zeros_like(a[0]) if k in pick else None for k in range(3)]
        s._chk(s.lib.hc_get_vertices(s.h, *[hc._dp(o) for o in out]))
        for k in pick:
            assert np.array_equal(out[k], a[k])
    s.set_repulsion_force(a[1])
    assert np.array_equal(s.repulsion_force(), a[1])
    s.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_force_field_before_and_after_a_step(precision):
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
    s = _sim((33, 31, 35), precision)
    s.set_force_limit(u.f_limit)
    s.add_cells(s.add_cell_type(model, v, t, p, inner), cases.place(v, (16, 15, 17))[None])
    f = np.random.default_rng(1).normal(size=(len(v), 3)) * 0.01 * u.f_limit
    s.set_vertices(f=f)
    s.stage("spread")
    F = s.force_field()
    assert np.allclose(F.sum(1), f.sum(0), rtol=1e-5 if precision else 1e-11, atol=1e-7 * np.abs(f).sum())
    s.step(2)
    assert not s.force_field().any()
    s.close()
