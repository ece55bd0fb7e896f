"""Total and insertion energies on both sides of the lines between the numbers of
lanes per query: within the bound on the summation order of the oracle's, infinite
where it is, and hard overlaps found wherever they are."""
import numpy as np
import pytest

import _oracle as O
import _pkg
from test_gpu_forms import _lattice

pytestmark = pytest.mark.gpu

LJ, OP = (1.0, 1.0, 2.5, 2.5), (10000.0, 0.2, 100.0, 1.0)


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.mark.parametrize("model,params,density,dim,ns", [
    ("lj_shifted", LJ, 0.8, 3, (65536, 65537, 98304, 98305)),       # 32, 8, 8 and 2 lanes
    ("lj_shifted", LJ, 0.05, 3, (16384, 16385, 98304, 98305)),      # 32, 8, 8 and 1
    ("lj_shifted", LJ, 0.7, 2, (16384, 16385, 98304, 98305)),
    ("overlap_penalty", OP, 0.9, 3, (16385, 98305))])
def test_total_energy(hmc, model, params, density, dim, ns):
    for n in ns:
        L = np.full(dim, (n / density) ** (1.0 / dim)) * np.array([1.02, 1.0, 1 / 1.02])[:dim]
        pos = _lattice(L, n, jitter=0.1)
        ref = O.OracleSystem(L, pos, model=model, params=params)
        sim = hmc.GpuParallelSweep(L, pos, model=model, params=params)
        want = ref.total_energy()
        for e, bound in (sim.total_energy(), sim.total_energy_noalloc()):
            assert abs(e - want) <= bound and bound < 1e-6 * max(abs(want), 1.0), (n, e, want, bound)
        sim.close()


@pytest.mark.parametrize("n", [16384, 98304, 98305])
def test_hard_overlap(hmc, n):
    L = np.full(3, (n / 0.5) ** (1.0 / 3.0))
    pos = _lattice(L, n)
    for i in (0, n // 2, n - 1):
        bad = pos.copy()
        bad[i] = pos[i - 1] + np.array([0.3, 0.0, 0.0])
        sim = hmc.GpuParallelSweep(L, bad)
        assert sim.total_energy()[0] == np.inf
        sim.set_positions(pos)
        assert sim.total_energy()[0] == 0.0
        sim.close()


@pytest.mark.parametrize("n", [32767, 32768, 32769])
def test_insertions(hmc, n):
    L = np.array([12.0, 13.0, 14.0])
    pos = _lattice(L, 300, jitter=0.2)
    ref = O.OracleSystem(L, pos, model="lj_shifted", params=LJ)
    sim = hmc.GpuParallelSweep(L, pos, model="lj_shifted", params=LJ)
    cand = np.random.default_rng(2).uniform(-0.5, 0.5, (n, 3)) * L
    e, bound = sim.delta_energy_insert(cand)
    sim.close()
    want = np.array([ref.delta_energy_insert(c) for c in cand])
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(e), inf)
    assert (np.abs(e[~inf] - want[~inf]) <= bound[~inf]).all()
