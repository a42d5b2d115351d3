"""The velocity field filled on the cells' support boxes only: cells on periodic corners, beside closed faces and
overlapping boxes, stepped alone and in a batch, against the FP64 oracle; and a cell without a finite box beside a
good one, which steps as if it were alone."""
import numpy as np
import pytest

import cases
from oracle import OracleSim

pytestmark = pytest.mark.gpu

CENTRES = [(20.3, 18.7, 22.1), (0.2, 39.6, 20.0), (21.5, 20.1, 43.9), (26.0, 18.0, 23.0)]


def _make(kind, centres, periodic, sim=None, precision=0):
    import hemocell_amd as hc
    u = cases.units()
    model, v, t, p, inner = cases.mesh(kind, u, hc.build_mesh)
    n = (40, 40, 44)
    if sim is None:
        s = hc.Simulation(0)
        s.lattice_init(*n, u.tau, periodic=periodic, precision=precision)
    else:
        s = OracleSim(*n, u.tau, periodic=periodic)
    s.init_equilibrium(1.0, [2e-3, 1e-3, -1e-3])
    s.set_force_limit(u.f_limit)
    rng = np.random.default_rng(5)
    d = v - v.mean(axis=0)
    x = np.stack([d @ (np.eye(3) + np.diag(0.02 * rng.uniform(-1, 1, 3))) + c for c in centres])
    s.add_cells(s.add_cell_type(model, v, t, p, inner), x)
    return s, x


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["RBC", "PLT", "WBC"])
def test_alone_and_in_a_batch(kind, precision):
    import hemocell_amd as hc
    setups = [(CENTRES[:1], (1, 1, 1)), (CENTRES[1:3], (1, 1, 1)), (CENTRES[:1] + CENTRES[3:], (0, 1, 0))]
    sims = [_make(kind, c, p, precision=precision)[0] for c, p in setups]
    hc.step_batch(sims, 3)
    for s, (c, p) in zip(sims, setups):
        o, x = _make(kind, c, p, sim="oracle")
        o.step(3)
        a, _ = _make(kind, c, p, precision=precision)
        a.step(3)
        for got in (s.vertices(), a.vertices()):
            e = max(cases.rel_l2(got[0] - x.reshape(-1, 3), o.vertices()[0] - x.reshape(-1, 3)),
                    cases.rel_l2(got[1], o.vertices()[1]))
            assert e < (2e-5 if precision else 1e-10), (kind, c, p, e)
        s.close()
        a.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_a_cell_without_a_box(precision):
    alone, _ = _make("PLT", CENTRES[:1], (1, 1, 1), precision=precision)
    alone.step(4)
    s, x = _make("PLT", [CENTRES[0], (5.0, 5.0, 5.0)], (1, 1, 1), precision=precision)
    nv = x.shape[1]
    x = x.reshape(-1, 3)
    x[nv + 3] = np.nan
    s.set_vertices(x=x)
    s.step(4)
    for got, want in zip(s.vertices(), alone.vertices()):
        assert np.allclose(got[:nv], want, rtol=1e-6 if precision else 1e-12, atol=0.0)
    s.close()
    alone.close()
