"""Bodies that do not fill the box: the applies' plan follows the state, with the
same moves as one launch per colour before and after it does."""
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


def _compare(hmc, L, pos, d, kT, by_steps, **kw):
    """Runs both forms; returns the persistent one's form and its stats after each call."""
    a = hmc.GpuParallelSweep(L, pos, **kw)
    b = hmc.GpuParallelSweep(L, pos, persistent=False, **kw)
    seen, step = [(a.debug_form(), a.stats())], 0
    for n in by_steps:
        if n == 1:
            assert a.apply(step, 0, 5, kT, d) == b.apply(step, 0, 5, kT, d)
        else:
            assert a.run(step, 5, kT, d, n) == b.run(step, 5, kT, d, n)
        step += n
        for x, y in zip(a.positions(), b.positions()):
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64))
        seen.append((a.debug_form(), a.stats()))
    a.close()
    b.close()
    return seen


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("by_steps", [(1, 1, 1), (5, 3)])
@pytest.mark.parametrize("n,factor,width", [
    (2000, (2.0, 2.0, 2.0), 1.0), (2000, (4.0, 4.0, 4.0), 1.3), (20000, (1.0, 1.0, 6.0), 1.0), (2300, (3.0, 3.0), 2.0)])
def test_regions_of_a_drop(hmc, n, factor, width, by_steps, precision):
    dim = len(factor)
    a = (n / 0.85) ** (1.0 / dim)
    drop = a * np.array([1.0, 1.01, 0.99])[:dim]
    seen = _compare(hmc, drop * np.array(factor), _lattice(drop, n, jitter=0.01), 0.05, 1.0, by_steps,
                    precision=precision, body_interaction_range=width)
    over = [s["tile_overflows"] for _, s in seen]
    # the first apply runs over the boxes' capacity, none after the second plan at most
    assert all(f["persistent"] for f, _ in seen)
    assert over[1] > 0 and over[-1] <= 2 * over[1] and (by_steps[0] > 1 or over[-1] == over[-2])


def test_a_drop_too_dense_for_regions(hmc):
    # FP64: regions for the mean density, none whose boxes hold the drop
    n = 20000
    a = (n / 0.85) ** (1.0 / 3.0)
    drop = a * np.array([1.0, 1.01, 0.99])
    seen = _compare(hmc, 4.0 * drop, _lattice(drop, n, jitter=0.01), 0.05, 1.0, (1, 4), precision="fp64",
                    body_interaction_range=1.3)
    assert seen[0][0]["persistent"] == 1 and seen[1][0]["persistent"] == seen[2][0]["persistent"] == 0


def test_lanes_of_a_drop(hmc):
    # LJ: 337 candidates per trial, 5 by the mean density; then a gas of the same bodies
    n = 8000
    a = (n / 0.8) ** (1.0 / 3.0)
    drop = a * np.array([1.0, 1.01, 0.99])
    L = 4.0 * drop
    seen = _compare(hmc, L, _lattice(drop, n, jitter=0.05), 0.1, 0.7, (1, 3), model="lj_shifted")
    assert seen[0][0]["iso_lanes"] < 64 and seen[1][0]["iso_lanes"] == seen[2][0]["iso_lanes"] == 64
    sim = hmc.GpuParallelSweep(L, _lattice(drop, n, jitter=0.05), model="lj_shifted")
    sim.run(0, 5, 0.7, 0.1, 2)
    assert sim.debug_form()["iso_lanes"] == 64
    sim.set_positions(_lattice(L, n, jitter=0.05))
    sim.run(2, 5, 0.7, 0.1, 2)
    assert sim.debug_form() == seen[0][0]
    sim.close()
