"""The scale distribution function at the edges of its blocks and counters: runs
of 512 bodies, counters in LDS and beyond what is summed there (8192 bins), three
spaces along an axis, two, scans of two spaces, and overlaps."""
import numpy as np
import pytest

import _oracle as O
import _pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def _random(n, L, seed):
    # bodies of a cubic or square lattice, displaced by up to a fifth of its constant
    rng = np.random.default_rng(seed)
    d = len(L)
    m = np.ceil((n / np.prod(L)) ** (1.0 / d) * np.asarray(L)).astype(int)
    g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, d)
    g = g[rng.permutation(len(g))[:n]]
    a = np.asarray(L) / m
    return (g + 0.5) * a - np.asarray(L) / 2 + rng.uniform(-0.2, 0.2, (n, d)) * a


@pytest.mark.parametrize("L,n,xmax,nbins", [
    ((10.0, 9.0, 9.5), 511, 0.02, 200), ((10.0, 9.0, 9.5), 512, 0.02, 200), ((10.0, 9.0, 9.5), 513, 0.02, 1),
    ((40.0, 37.0, 41.0), 50000, 0.02, 8192), ((40.0, 37.0, 41.0), 50000, 0.02, 8193),
    ((40.0, 37.0, 41.0), 50000, 0.4, 1000),
    ((3.5, 6.3, 12.2), 150, 0.1, 50), ((2.6, 2.7, 30.0), 100, 0.1, 50), ((6.0, 6.0, 6.0), 100, 0.3, 64),
    ((50.0, 31.0), 1500, 0.1, 100), ((4.0, 60.0), 200, 0.2, 100)])
def test_sdf_counts(hmc, L, n, xmax, nbins):
    L = np.array(L)
    sim = hmc.GpuParallelSweep(L, _random(n, L, 5))
    h, ov = sim.sdf(xmax, xmax / nbins, nbins=nbins)
    _, s = sim.positions()
    want, wov = O.sdf(L, s, 1.0, xmax, xmax / nbins, nbins)
    assert np.array_equal(h, want) and ov == wov
    sim.close()
