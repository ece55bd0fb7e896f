"""All lengths scaled by a power of two, far from 1 and beyond the range of FP32: every
FP64 operation scales exactly, so the moves and counts are those of the unscaled
system.  (Mixed precision at scales whose squares FP32 holds.)"""
import numpy as np
import pytest

import _pkg
from test_gpu_forms import _lattice

pytestmark = pytest.mark.gpu

CUBE = np.array([[a, b, c] for a in (-0.5, 0.5) for b in (-0.5, 0.5) for c in (-0.5, 0.5)])


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def _bits(sim, scale):
    return np.concatenate([(x / scale).ravel() for x in sim.positions()]).view(np.uint64)


@pytest.mark.parametrize("precision,power", [("fp64", p) for p in (-140, -70, -41, 25, 30, 41, 63, 66, 140)] +
                         [("mixed", p) for p in (-45, -30, 25, 30, 45)])
@pytest.mark.parametrize("L,n", [((25.2, 26.3, 27.1), 9000), ((61.2, 62.3), 2300), ((4.1, 4.3, 4.2), 30)])
def test_hard_shapes(hmc, L, n, precision, power):
    pos, out = _lattice(np.array(L), n), []
    for f in (1.0, 2.0**power):
        sim = hmc.GpuParallelSweep(np.array(L) * f, pos * f, diameter=f, precision=precision)
        cnt = sim.run(0, 3, 1.0, 0.12 * f, 3)
        hist, ov = sim.sdf()
        out.append((cnt, ov, hist.tolist(), _bits(sim, f)))
        sim.close()
    assert out[0][:3] == out[1][:3] and np.array_equal(out[0][3], out[1][3])


@pytest.mark.parametrize("precision,power", [("fp64", p) for p in (-140, -70, 41, 63, 66, 140)] +
                         [("mixed", p) for p in (-140, -80, -45, -30, 30, 45, 66, 140)])
@pytest.mark.parametrize("L,n", [((36.2, 31.1, 35.3), 25000), ((10.1, 10.2, 10.3), 700), ((60.3, 72.1), 2400)])
def test_lennard_jones(hmc, L, n, precision, power):
    pos, out = _lattice(np.array(L), n, jitter=0.1), []
    for f in (1.0, 2.0**power):
        sim = hmc.GpuParallelSweep(np.array(L) * f, pos * f, model="lj_shifted", params=(1.0, f, 2.5 * f, 2.5 * f),
                                   precision=precision)
        out.append((sim.run(0, 3, 1.2, 0.12 * f, 2), _bits(sim, f)))
        sim.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("power", [-140, -70, 66, 140])
def test_overlap_penalty(hmc, power):
    L = np.array([20.1, 21.2, 22.3])
    pos, out = _lattice(L, 8000, jitter=0.3), []
    for f in (1.0, 2.0**power):
        sim = hmc.GpuParallelSweep(L * f, pos * f, model="overlap_penalty", params=(1e4 / f / f, 0.2 * f, 100.0, f))
        out.append((sim.run(0, 3, 1.0, 0.1 * f, 3), _bits(sim, f)))
        sim.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("power", [30, 64, 140])
def test_cubes(hmc, precision, power):
    L = np.array([15.0, 15.1, 16.2])
    pos, out = _lattice(L, 12 * 12 * 13, jitter=0.0), []
    for f in (1.0, 2.0**power):
        sim = hmc.GpuParallelSweep(L * f, pos * f, model="convex", vertices=CUBE * f, precision=precision)
        cnt = sim.run_moves(0, 3, 1.0, [("translate", 0.05 * f), ("rotate", 0.1)], 3)
        out.append((cnt, _bits(sim, f)))
        sim.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


def test_batch(hmc):
    for power in (-45, 30, 45):
        out = []
        for f in (1.0, 2.0**power):
            systems = [(np.array([12.2 + r, 13.3, 14.1]) * f, _lattice(np.array([12.2 + r, 13.3, 14.1]), 1200) * f, None)
                       for r in range(4)]
            b = hmc.GpuBatch(systems, diameter=f, precision="mixed")
            cnt = b.run(0, np.arange(4), 1.0, 0.1 * f, 3)
            out.append((cnt, np.concatenate([(x / f).ravel() for r in range(4) for x in b.positions(r)]).view(np.uint64)))
            b.close()
        assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
