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
