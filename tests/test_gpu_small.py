"""Small FP64 systems with isotropic pair energies, whose applies one workgroup
runs from LDS: replays against the oracle at the fewest spaces, in flat boxes,
with empty spaces, with one body, and on both sides of the largest system taken."""
import numpy as np
import pytest

import _pkg
from test_gpu_lj import _replay_lj

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.fixture(scope="module")
def wl():
    return _pkg.workloads()


def _random(n, L, seed, scale=0.9):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / len(L))))
    g = np.stack(np.meshgrid(*[np.arange(m)] * len(L), indexing="ij"), -1).reshape(-1, len(L))
    g = g[rng.permutation(len(g))[:n]]
    a = np.asarray(L) / m
    return (g + 0.5) * a - np.asarray(L) / 2 + rng.uniform(-0.1, 0.1, (n, len(L))) * a * scale


@pytest.mark.parametrize("L,n,model,params", [
    ((5.3, 5.2, 5.4), 60, "lj_shifted", (1.0, 1.0, 2.5, 2.5)),      # two spaces per axis: four wavefronts per trial
    ((5.2, 10.4, 15.5), 300, "lj_shifted", (1.0, 1.0, 2.5, 2.5)),   # 2 x 4 x 6 spaces
    ((10.1, 10.2, 10.3), 700, "lj", (1.0, 1.0, 2.5)),               # two wavefronts per trial
    ((10.0, 10.0, 10.0), 5, "lj", (1.0, 1.0, 2.5)),                 # most spaces empty, spaces as wide as the cutoff
    ((10.1, 10.2, 10.3), 1, "lj", (1.0, 1.0, 2.5)),                 # a single body
    ((15.5, 15.4, 15.3), 1100, "lj_shifted", (1.0, 1.0, 2.5, 2.5)),  # 27 trials a pass: rounds of 16
    ((5.3, 5.2), 14, "lj", (1.0, 1.0, 2.5)),                        # 2D, two spaces per axis
    ((20.5, 5.2), 60, "lj_shifted", (1.0, 1.0, 2.5, 2.5)),          # 2D, 8 x 2
    ((40.5, 40.2), 700, "lj", (1.0, 1.0, 2.5)),                     # 2D, 64 trials a pass
    ((6.3, 6.2, 6.1), 130, "overlap_penalty", (10000.0, 0.2, 100.0, 1.0)),
    ((9.3, 8.2, 10.1), 400, "overlap_penalty", (5.0, 0.9, 0.3, 1.0)),
])
def test_small_replays(hmc, wl, L, n, model, params):
    pos = _random(n, L, 7)
    _replay_lj(hmc, np.array(L), pos, model, params, 1.2, 0.2, 8, seed=11)


@pytest.mark.parametrize("n", [1370, 1420, 1700])
def test_largest_small_system_and_the_next(hmc, wl, n):
    # about 1,400 bodies fill the LDS; the next sizes run the per-colour passes
    L = np.array([13.0, 13.0, 13.0])
    _replay_lj(hmc, L, _random(n, L, 3), "lj_shifted", (1.0, 1.0, 2.5, 2.5), 1.2, 0.1, 2, seed=5)
