"""The device's order of persistent launches never names a stream whose steps are
captured in graphs: a batch, or a context, that gives its persistent form up leaves it."""
import threading

import numpy as np
import pytest

import _pkg
from test_gpu_forms import _lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def _batch(hmc):
    L = np.array([14.3, 15.2, 40.3])
    systems = [(L, _lattice(L, 8000), None), (L, _lattice(L, 7000), None)]
    return hmc.GpuBatch(systems, precision="mixed"), systems


def _pile(hmc, b, systems):
    # all bodies of a replica in a few spaces: no region's box holds them
    n = len(systems[0][1])
    b.set_positions(0, np.random.default_rng(1).uniform(-0.4, 0.4, (n, 3)))


def test_a_batch_without_regions_leaves_the_order(hmc):
    b, systems = _batch(hmc)
    seeds = np.arange(2)
    b.run(0, seeds, 1.0, 0.1, 2)
    assert b.stats(0)["tiled"] == 2 and hmc.lib().hmc_debug_order(0) == 1
    _pile(hmc, b, systems)
    b.run(2, seeds, 1.0, 0.1, 1)
    assert b.stats(0)["tiled"] == 1 and hmc.lib().hmc_debug_order(0) == 0
    b.close()


def test_a_context_that_gives_way_leaves_the_order(hmc):
    L = np.array([14.3, 15.2, 16.3])
    pos = _lattice(L, 2500)
    sim = hmc.GpuParallelSweep(L, pos, precision="mixed")
    sim.run(0, 1, 1.0, 0.1, 2)
    assert hmc.lib().hmc_debug_order(0) == 1
    sim.set_positions(pos, np.roll(pos, 1, axis=0))  # sites away from their bodies
    assert sim.debug_form()["persistent"] == 0 and hmc.lib().hmc_debug_order(0) == 0
    sim.close()


def test_captures_beside_persistent_launches(hmc):
    b, systems = _batch(hmc)
    seeds = np.arange(2)
    b.run(0, seeds, 1.0, 0.1, 2)
    _pile(hmc, b, systems)
    L = np.array([14.3, 15.2, 16.3])
    sim = hmc.GpuParallelSweep(L, _lattice(L, 2500), precision="mixed")
    errors = []

    def captures():
        try:
            for k in range(6):
                b.set_positions(1, systems[1][1])
                b.run(2 + 4 * k, seeds, 1.0, 0.1, 4)
        except Exception as e:
            errors.append(e)

    def launches():
        try:
            for k in range(60):
                sim.run(4 * k, 1, 1.0, 0.1, 4)
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=f) for f in (captures, launches)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    b.close()
    sim.close()
