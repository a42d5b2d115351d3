"""The autotuner tries what a context runs with before any other launch shape and keeps it unless another is faster."""
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", [("RBC",), ("RBC", "WBC2562"), ("WBC",)])
@pytest.mark.parametrize("precision", [0, 1])
def test_untuned_shapes_are_candidates(kinds, precision):
    import hemocell_amd as hc
    u = cases.units()
    s = hc.Simulation(0)
    s.lattice_init(48, 48, 48, u.tau, precision=precision)
    s.init_equilibrium(1.0, [1e-3, 0, 2e-3])
    s.set_force_limit(u.f_limit)
    for kind, at in zip(kinds, ([(12, 12, 12), (12, 36, 12), (36, 12, 36), (12, 12, 36), (36, 36, 10)], [(32, 32, 32)])):
        model, v, t, p, inner = cases.mesh(kind, u, hc.build_mesh)
        s.add_cells(s.add_cell_type(model, v, t, p, inner), [cases.place(v, c) for c in at])
    rep = s.autotune(3)
    assert next(iter(rep["spread_box_bytes"])) == "0"
    assert "RBC" not in kinds or next(iter(rep["rbc_threads"])) == "0"
    again = s.autotune(3)
    s.close()
    for r in list(rep.values()) + list(again.values()):
        trials = {k: ms for k, ms in r.items() if k != "chosen"}
        first, chosen = next(iter(trials)), str(r["chosen"])
        # times are reported with six digits
        assert chosen == first or trials[chosen] < 0.99 * trials[first] * (1 + 1e-5)
    for name in set(rep) & set(again):
        assert next(iter(again[name])) == str(rep[name]["chosen"])
