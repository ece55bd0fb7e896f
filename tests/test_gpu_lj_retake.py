"""The FP64 re-take of an LJ trial with more bodies within the cutoff than its list holds
(768), in regions whose boxes still fit their LDS."""
import numpy as np
import pytest

import _pkg
from test_gpu_lj import _replay_lj

pytestmark = pytest.mark.gpu

LJ = (1.0, 1.0, 2.5, 2.5)


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def test_a_cluster_in_a_hollow(hmc):
    # 860 bodies within 2.3 of one another, nothing else within 18 of them (so that a box
    # of 15 with the cluster holds no more), and bodies whose boxes hold about 790
    rng = np.random.default_rng(5)
    L = np.array([80.9, 80.8, 81.0])
    bg = rng.uniform(-0.5, 0.5, (120000, 3)) * L
    bg = bg[np.abs(bg).max(axis=1) > 18.0]
    u = rng.normal(size=(860, 3))
    u *= (1.15 * rng.uniform(0.02, 1.0, 860) ** (1.0 / 3.0) / np.linalg.norm(u, axis=1))[:, None]
    d2 = ((u[:, None] - u[None]) ** 2).sum(-1)
    # a cluster space holds no other body, so its trial is of one of these; moves of 0.05
    # leave all of them within the cutoff
    assert (np.sqrt(d2).max() < 2.5 - 4 * 0.05) and len(u) - 1 > 768
    st, _ = _replay_lj(hmc, L, np.concatenate([bg, u]), "lj_shifted", LJ, 1.2, 0.05, 2, seed=2, precision="mixed",
                       trace=False)
    assert st["tiled"] == 2 and st["tile_overflows"] == 0 and st["band_retests"] > 0
