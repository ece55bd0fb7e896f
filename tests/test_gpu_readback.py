"""Reads of device state through pinned chunks: sizes on both sides of a chunk
(131,072 words), of two and of three, with either output left out, and the
positions of each replica of a batch."""
import numpy as np
import pytest

import _pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.mark.parametrize("dim,n", [(3, 1), (3, 21845), (3, 21846), (3, 43690), (3, 43691), (3, 65537), (2, 32768), (2, 32769)])
def test_positions_return_what_was_set(hmc, dim, n):
    rng = np.random.default_rng(n)
    L = np.full(dim, 100.0)
    b = rng.uniform(-50.0, 50.0, (n, dim))
    s = rng.uniform(-50.0, 50.0, (n, dim))
    sim = hmc.GpuParallelSweep(L, b, sites=s)
    gb, gs = sim.positions()
    assert np.array_equal(gb, b) and np.array_equal(gs, s)
    for want, out in ((b, 0), (s, 1)):
        x = np.zeros((n, dim))
        p = [None, None]
        p[out] = hmc._p(x)
        assert hmc.lib().hmc_get_state(sim.h, *p) == 0
        assert np.array_equal(x, want)
    assert hmc.lib().hmc_get_state(sim.h, None, None) == 0
    sim.close()


@pytest.mark.parametrize("n", [16384, 16385])
def test_orientations_return_what_was_set(hmc, n):
    rng = np.random.default_rng(n)
    wl = _pkg.workloads()
    b = rng.uniform(-50.0, 50.0, (n, 3))
    q, u = rng.normal(size=(n, 4)), rng.normal(size=(n, 4))
    sim = hmc.GpuParallelSweep(np.full(3, 100.0), b, model="convex", vertices=wl.UNIT_CUBE, orientations=q, site_orientations=u)
    gq, gu = sim.orientations()
    assert np.array_equal(gq, q) and np.array_equal(gu, u)
    sim.close()


def test_batch_positions_return_what_was_set(hmc):
    rng = np.random.default_rng(3)
    systems = [(np.full(3, 60.0), rng.uniform(-30.0, 30.0, (n, 3)), None) for n in (1, 4, 21846, 500, 50000)]
    sim = hmc.GpuBatch(systems)
    for r, (_, b, _) in enumerate(systems):
        assert np.array_equal(sim.positions(r)[0], b)
    sim.close()
