"""With the exact spread a cell ends in the same bits however its launch lays out its positions: staged, in LDS only, or
in global memory beside many red cells and in the persistent launch; alone and in a batch."""
import numpy as np
import pytest

import cases
import geodesic

pytestmark = pytest.mark.gpu


def _sim(monkeypatch, frequency, mixed):
    import hemocell_amd as hc
    monkeypatch.setenv("HC_MIXED", mixed)
    u = cases.units()
    s = hc.Simulation(0)
    s.lattice_init(126, 126, 126, u.tau, precision=0)
    s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
    s.set_force_limit(u.f_limit)
    s.set_exact_spread(True)
    centres = 18 * (np.stack(np.meshgrid(*[np.arange(7)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5)
    v, t = geodesic.sphere(frequency, 8.0)
    for kind, at in (("RBC", centres[:256]), ("WBC", centres[-1:])):
        model, w, wt, p, inner = cases.mesh(kind, u, hc.build_mesh)
        if kind == "WBC":
            w, wt, inner = v, t, np.array([(a, int(((v + v[a]) ** 2).sum(1).argmin())) for a in range(0, len(v), 7)],
                                          dtype=np.int32)
        d = (w - w.mean(axis=0)) * (1.02, 0.99, 0.99)
        s.add_cells(s.add_cell_type(model, w, wt, p, inner), np.stack([d + c for c in at]))
    return s


# 1442 and 1962 vertices: from 1366 on positions stay in global memory as a side type's, up to 2190 they can be staged;
# 642: staged, but for the persistent launch
@pytest.mark.parametrize("frequency", [8, 12, 14])
def test_launches_agree(monkeypatch, frequency):
    import hemocell_amd as hc
    out = []
    for how in ("alone", "in LDS", "persistent", "batch"):
        monkeypatch.setenv("HC_SIDE_GPOS", "0" if how == "in LDS" else "1")
        s = _sim(monkeypatch, frequency, "1" if how == "persistent" else "0")
        if how == "batch":
            hc.step_batch([s], 6)
        else:
            s.step(6)
        out.append(s.vertices() + (s.populations(),))
        s.close()
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)
