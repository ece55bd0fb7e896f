"""Neighbour rows of a site on the periodic end of the checkerboard: an ulp below
origin + L, where the space index x - origin over the width rounds up to the
number of spaces and the site belongs to the first space."""
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


def _draws(step, seed, dim):
    """The origin draws of the checkerboard of counter (step, 0, seed)."""
    return O.sample(step, 0, seed, 2**64 - 1, "f64", dim)


def _end(L, k, u):
    """A coordinate whose body and site lie below origin + L but in space 0 of k
    along an edge of L, with the draw u; None if this edge has none."""
    w = L / k
    o = -L / 2.0 - u * w
    x = o + L
    for _ in range(8):
        x = np.nextafter(x, -np.inf)
    for _ in range(12):
        lam = x / L
        s = (lam - np.round(lam)) * L
        if all(y - o < L and np.floor((y - o) / w) == k for y in (x, s)):
            return x
        x = np.nextafter(x, np.inf)
    return None


def _edges(k, width, u, rng):
    """Edges a little over k[a] widths that have such a coordinate, and it."""
    L, x = [], []
    for ka, ua in zip(k, u):
        xa = None
        for _ in range(100000):
            La = width * (ka + 0.9 * rng.random())
            xa = _end(La, ka, ua)
            if xa is not None:
                break
        assert xa is not None
        L.append(La)
        x.append(xa)
    return np.array(L), np.array(x)


def _wrap(L, x):
    return x - L * np.round(x / L)


@pytest.mark.parametrize("k", [(5, 6, 7), (9, 10, 6), (12, 9)])
def test_sdf_finds_the_neighbour_across_the_end(hmc, k):
    xmax, nbins, D = 0.1, 100, len(k)
    L, x = _edges(k, 1.0 / (1.0 - xmax) * (1.0 + 2.0**-28), _draws(0, 0, D), np.random.default_rng(3))
    far = x + L / 2.0  # a third body, near neither
    for axis in range(D):
        step = np.zeros(D)
        step[axis] = 1.02
        pos = np.stack([x, _wrap(L, x - step), _wrap(L, far)])
        pos[0] = x  # (not wrapped again)
        sim = hmc.GpuParallelSweep(L, pos)
        h, ov = sim.sdf(xmax, xmax / nbins, nbins=nbins)
        want, wov = O.sdf(L, pos, 1.0, xmax, xmax / nbins, nbins, all_pairs=True)
        assert want.sum() == 2
        assert np.array_equal(h, want) and ov == wov
        sim.close()
