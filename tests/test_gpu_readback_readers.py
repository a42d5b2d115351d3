"""Large read-backs (64 MB and more), which several host threads share: just below, at and above that size, and counts
that do not divide evenly; what was set comes back bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 64 MB are 441505.7 nodes of 19 populations
@pytest.mark.parametrize("shape", [(441505, 1, 1), (441506, 1, 1), (441507, 1, 1), (97, 89, 61)])
def test_populations(shape):
    import hemocell_amd as hc
    s = hc.Simulation(0)
    s.lattice_init(*shape, 1.1, periodic=(1, 1, 1))
    f = np.random.default_rng(3).uniform(-1e-2, 1e-2, size=(19, int(np.prod(shape))))
    s.set_populations(f)
    assert np.array_equal(s.populations(), f)
    s.close()


def test_two_contexts_at_once():
    import threading

    import hemocell_amd as hc
    sims, want, got = [], [], [None] * 2
    for k in range(2):
        s = hc.Simulation(0)
        s.lattice_init(80, 81, 82, 1.1, periodic=(1, 1, 1))
        want.append(np.random.default_rng(k).uniform(-1e-2, 1e-2, size=(19, 80 * 81 * 82)))
        s.set_populations(want[k])
        sims.append(s)

    def read(k):
        got[k] = sims[k].populations()

    threads = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert np.array_equal(got[k], want[k])
        sims[k].close()
