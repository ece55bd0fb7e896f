"""The persistent apply for hard convex polyhedra and the rows of neighbour
spaces behind it, at their edges: two, four and six spaces per axis, ragged
last regions, one region in all, and the sizes beyond which one launch per
colour takes over.  Replays are compared with the oracle bit for bit (trace,
counts, positions, orientations), the two forms with each other."""
import sys

import numpy as np
import pytest

import _oracle as O
import _pkg
from test_gpu_convex import TETRA, _replay

pytestmark = pytest.mark.gpu


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def _box(n, phi, vol=1.0):
    a = (vol / phi) ** (1.0 / 3.0)
    i, j, k = np.meshgrid(*[np.arange(x) for x in n], indexing="ij")
    L = np.array(n) * a
    return L, (np.stack([i.ravel(), j.ravel(), k.ravel()], 1) + 0.5) * a - L / 2, np.tile([1.0, 0, 0, 0], (int(np.prod(n)), 1))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,phi", [((4, 4, 4), 0.50), ((4, 6, 9), 0.55), ((9, 4, 6), 0.40), ((12, 5, 16), 0.55),
                                   ((7, 18, 9), 0.30)])
def test_replay_shapes(hmc, n, phi, precision):
    L, pos, q = _box(n, phi)
    _replay(hmc, L, pos, q, O.CUBE, 0.08, 0.2, 6, precision=precision)


def test_replay_dilute_with_long_moves(hmc):
    L, pos, q = _box((5, 7, 8), 0.05, vol=1.0 / 3.0)
    _replay(hmc, L, pos, q, TETRA, 0.9, 1.5, 6)


@pytest.mark.parametrize("n,phi,persistent", [((24, 24, 24), 0.55, True), ((50, 50, 50), 0.30, True),
                                              ((64, 64, 64), 0.30, False)])
def test_both_forms_agree(hmc, n, phi, persistent):
    L, pos, q = _box(n, phi)
    out = []
    for per_colour in (False, True):
        sim = hmc.GpuParallelSweep(L, pos, model="convex", vertices=O.CUBE, orientations=q, persistent=not per_colour)
        counts = sim.run_moves(0, 3, 1.0, [("translate", 0.08), ("rotate", 0.2)], 4)
        s = sim.stats()
        assert (s["regions"] > 0) == (persistent and not per_colour)
        out.append([np.concatenate([x.ravel() for x in sim.positions() + sim.orientations()]), counts])
        log(f"{n} phi {phi}: {s['regions']} regions of {s['tile_shape']}")
        sim.close()
    assert np.array_equal(out[0][0].view(np.uint64), out[1][0].view(np.uint64))
    assert out[0][1:] == out[1][1:]
