"""Energies and kT scaled alike by a power of two, far beyond the range of FP32: every
FP64 operation scales exactly, so the moves are those of the unscaled system."""
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


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("L,n", [((10.1, 10.2, 10.3), 700), ((36.2, 31.1, 35.3), 25000), ((60.3, 72.1), 2400)])
@pytest.mark.parametrize("power", [130, 127, 125, -125, -140])
def test_moves_do_not_change(hmc, L, n, precision, power):
    pos = _lattice(np.array(L), n, jitter=0.1)
    out = []
    for scale in (1.0, 2.0**power):
        sim = hmc.GpuParallelSweep(np.array(L), pos, model="lj_shifted", params=(scale, 1.0, 2.5, 2.5),
                                   precision=precision)
        counts = [sim.apply(k, 0, 4, 1.2 * scale, 0.12) for k in range(2)]
        out.append((counts, np.concatenate([x.ravel() for x in sim.positions()]).view(np.uint64)))
        sim.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
