"""A vertex far outside a walled box with periodic axes: the fused step looks up the same wall nodes as the separate
passes, whatever the size of the (finite) position."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("far", [3e9, 4.6e15, 9.1e15, 7.7e17])
def test_wall_contact(monkeypatch, far, precision):
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
    out = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("HC_FUSE", fuse)
        s = hc.Simulation(0)
        # two thirds of the periodic planes are wall, so that about as many of the far vertices touch it
        mask = np.zeros((31, 24, 37), dtype=np.uint8)
        mask[:, 0] = mask[:, -1] = 1
        mask[::3, :4] = mask[1::3, :4] = 1
        s.lattice_init(31, 24, 37, u.tau, periodic=(1, 0, 1), node_type=mask.reshape(-1), precision=precision)
        s.init_equilibrium(1.0, [0, 0, 0])
        s.add_cells(s.add_cell_type(model, v, t, p, inner), cases.place(v, (15, 12, 18))[None])
        rng = np.random.default_rng(7)
        x = s.vertices()[0]
        k = np.arange(0, len(x), 5)
        x[k, 0] = np.floor(far * (1 + rng.uniform(0, 0.1, len(k)))) * rng.choice((-1, 1), len(k))
        x[k, 1] = 2.0
        x[k, 2] = np.floor(far * (1 + rng.uniform(0, 0.1, len(k))))
        s.set_vertices(x=x, v=np.zeros_like(x), f=np.zeros_like(x))
        s.step(1)
        out.append((s.removed_vertices(), s.wall_hits()))
        s.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    assert 0 < out[0][1] < len(k)


@pytest.mark.parametrize("precision", [0, 1])
# sizes of the support box whose product is 0 or negative in 64 bits
@pytest.mark.parametrize("size", [(2 ** 22, 2 ** 22, 2 ** 22), (2 ** 21, 2 ** 21, 2 ** 21), (2 ** 23, 2 ** 22, 2 ** 23),
                                  (2 ** 29, 2 ** 29, 2 ** 29)])
def test_spread_of_a_cell_across_the_axes(monkeypatch, size, precision):
    """A periodic box, a cell whose vertices lie millions of nodes apart: its spread by itself adds the same force as the
    spread by vertex."""
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh("RBC", u, hc.build_mesh)
    out = []
    for spread in ("vertex", "cell"):
        monkeypatch.setenv("HC_SPREAD", spread)
        s = hc.Simulation(0)
        s.lattice_init(31, 24, 37, u.tau, precision=precision)
        s.init_equilibrium(1.0, [0, 0, 0])
        s.set_force_limit(u.f_limit)
        s.add_cells(s.add_cell_type(model, v, t, p, inner), cases.place(v, (15, 12, 18))[None])
        x = s.vertices()[0]
        x[5] = (3.25, 4.5, 5.75)
        x[9] = x[5] + np.array(size) - 2
        x = np.clip(x, x[5], x[9])
        f = np.random.default_rng(3).uniform(-1e-5, 1e-5, x.shape)
        s.set_vertices(x=x, f=f)
        s.stage("spread")
        out.append(s.force_field())
        s.close()
    assert np.abs(out[0]).max() > 0 and cases.rel_l2(out[1], out[0]) < (1e-6 if precision else 1e-14)
