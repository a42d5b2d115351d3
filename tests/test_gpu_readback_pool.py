"""Read-backs share pinned slots: contexts opened one after another pin nothing anew, contexts read from several threads
at once get their own values."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mapped():
    """Bytes the process has mapped from the GPU's device node, pinned host memory among them."""
    total = 0
    for line in open("/proc/self/maps"):
        if "/dev/dri/" in line:
            low, high = line.split()[0].split("-")
            total += int(high, 16) - int(low, 16)
    return total


def _read(s):
    s.populations()
    s.fluid()
    s.fluid_stats()


def test_a_later_context_pins_nothing():
    import hemocell_amd as hc
    for first in (True, False):
        s = hc.Simulation(0)
        s.lattice_init(24, 25, 26, 1.1)
        s.init_equilibrium(1.0, [0, 0, 0])
        s.step(1)
        s.synchronize()
        before = _mapped()
        _read(s)
        assert first or _mapped() == before
        s.close()


def test_contexts_read_at_once():
    import hemocell_amd as hc
    sims, want, wrong = [], [], []
    for k in range(6):
        shape = (20 + 9 * k, 21, 22 + k)
        s = hc.Simulation(0)
        s.lattice_init(*shape, 1.1)
        want.append(np.random.default_rng(k).uniform(-1e-2, 1e-2, size=(19, int(np.prod(shape)))))
        s.set_populations(want[k])
        sims.append(s)

    def read(k):
        for _ in range(10):
            if not np.array_equal(sims[k].populations(), want[k]):
                wrong.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in sims:
        s.close()
    assert not wrong
