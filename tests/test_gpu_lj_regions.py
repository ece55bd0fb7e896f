"""The mixed-precision persistent LJ apply at the edges of how it shares out a
region's trials: one, two and four wavefronts, one to twelve trials, ragged last
regions, and an FP64 re-take of more bodies than its list holds.  Replays against
the oracle bit for bit."""
import numpy as np
import pytest

import _pkg
from test_gpu_lj import _replay_lj
from test_gpu_small import _random

pytestmark = pytest.mark.gpu

LJ = (1.0, 1.0, 2.5, 2.5)


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.mark.parametrize("L,n,threads", [
    ((15.3, 15.4, 15.5), 2400, 64),    # one trial of each colour per region
    ((20.4, 15.4, 15.5), 3200, 64),    # two
    ((20.4, 20.6, 15.5), 4100, 128),   # four
    ((20.4, 20.6, 20.9), 5600, 256),   # eight
    ((36.2, 31.1, 41.3), 30000, None),  # ragged regions
    ((41.0, 25.7, 15.6), 1000, None),   # empty spaces
    ((15.3, 15.4), 180, 64),
    ((62.3, 41.2), 2000, None),
])
def test_region_replays(hmc, L, n, threads):
    st, _ = _replay_lj(hmc, np.array(L), _random(n, L, 7), "lj_shifted", LJ, 1.2, 0.15, 3, seed=11, precision="mixed")
    assert st["tiled"] == 2 and st["tile_overflows"] == 0
    assert threads is None or st["region_threads"] == threads


def test_retake_of_more_bodies_than_its_list(hmc):
    # 850 bodies within the cutoff of one another (most pairs closer than the
    # FP32 bounds allow) in a dense box whose regions still hold them
    rng = np.random.default_rng(5)
    L = np.array([20.8, 20.8, 20.8])
    u = rng.normal(size=(850, 3))
    u *= (1.2 * rng.uniform(0.02, 1.0, 850) ** (1.0 / 3.0) / np.linalg.norm(u, axis=1))[:, None]
    pos = np.concatenate([_random(7500, L, 3), u])
    st, _ = _replay_lj(hmc, L, pos, "lj_shifted", LJ, 1.2, 0.05, 1, seed=2, precision="mixed")
    assert st["tiled"] == 2 and st["band_retests"] > 0
