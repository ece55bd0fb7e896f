"""Move sizes at the ends of FP64: a disk's displacement is a point of a square drawn until
it lies within the square of the move size, which none does where that is 0 or
infinite.  Such sizes are refused before anything is launched."""
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


@pytest.mark.parametrize("size", [1e-200, 1e-300, 5e-324, 1e155, 1e300, np.inf, np.nan, 0.0, -1.0])
def test_refused_in_2d(hmc, size):
    L = np.array([20.3, 21.2])
    for model in ("hard_sphere", "lj_shifted", "overlap_penalty"):
        sim = hmc.GpuParallelSweep(L, _lattice(L, 100), model=model)
        for call in (lambda: sim.apply(0, 0, 1, 1.0, size), lambda: sim.run(0, 1, 1.0, size, 2),
                     lambda: sim.run_moves(0, 1, 1.0, [("translate", 0.1), ("translate", size)], 2),
                     lambda: sim.tune_translate(0, 0, 1, 1.0, 0.2, 10, 1, size)):
            with pytest.raises(hmc.HmcError):
                call()
        sim.close()
    batch = hmc.GpuBatch([(L, _lattice(L, 100), None)] * 2)
    for call in (batch.run, lambda *a: batch.autotune(*a)):
        with pytest.raises(hmc.HmcError):
            call(0, np.arange(2), 1.0, np.array([0.1, size]), 2)
    batch.close()


@pytest.mark.parametrize("dim,sizes", [(2, (1e-150, 1e150)), (3, (1e-300, 1e300))])
def test_taken(hmc, dim, sizes):
    L = np.array([12.3, 13.2, 14.1])[:dim]
    for size in sizes:
        sim = hmc.GpuParallelSweep(L, _lattice(L, 80))
        acc, rej = sim.run(0, 1, 1.0, size, 2)
        assert acc + rej > 0 and (rej == 0 if size < 1.0 else True)
        sim.close()
