"""The two-kernel build of the persistent hard-shape applies: spaces of more
bodies than a bucket holds (8), at its edge and far beyond, in one scan block and
in several, with every body's turn and place as the oracle has it."""
import numpy as np
import pytest

import _pkg
from test_gpu_parity import _replay

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.fixture(scope="module")
def wl():
    return _pkg.workloads()


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("cells,extra", [((6, 6, 6), 7), ((6, 6, 6), 8), ((6, 6, 6), 9), ((14, 15, 16), 30)])
def test_spaces_of_many_bodies_3d(hmc, wl, cells, extra, precision):
    # `extra` bodies within 0.4 of one another, most of them in one space, in a
    # dilute box; the second such group straddles the periodic face
    L, pos = wl.fcc_spheres(cells, packing_fraction=0.25)
    rng = np.random.default_rng(4)
    a = rng.uniform(0.1, 0.5, (extra, 3))
    b = wl.wrap(L, L / 2 + rng.uniform(-0.2, 0.2, (extra, 3)))
    pos = np.concatenate([a, pos, b])[rng.permutation(len(pos) + 2 * extra)]
    _replay(hmc, L, pos, 0.2, 4, precision, seed=9)


@pytest.mark.parametrize("extra", [8, 9, 25])
def test_spaces_of_many_bodies_2d(hmc, extra):
    rng = np.random.default_rng(6)
    n, a = 40, 1.6
    i, j = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    L = np.array([n * a, n * a])
    pos = np.stack([(i.ravel() + 0.5) * a, (j.ravel() + 0.5) * a], 1) - L / 2
    pos = np.concatenate([pos, rng.uniform(0.1, 0.5, (extra, 2))])[rng.permutation(n * n + extra)]
    _replay(hmc, L, pos, 0.2, 4, "mixed", seed=3)


def test_one_body_and_none_to_spare(hmc):
    L = np.array([20.0, 20.0, 20.0])
    for n in (1, 2):
        pos = np.linspace(-8.0, 8.0, n)[:, None] * np.ones(3)
        _replay(hmc, L, pos, 0.2, 4, "mixed", seed=3)
