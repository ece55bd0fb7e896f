"""FP64 isotropic pair energies beyond the smallest systems: a group of lanes per
trial, in one persistent launch per apply or one launch per colour.  Replays
against the oracle at the edges: two spaces along an axis, rows across the
periodic face, scans of two spaces, empty spaces, spaces of many bodies, ragged
last regions, and every number of lanes; the two forms against each other."""
import numpy as np
import pytest

import _pkg
from test_gpu_lj import _replay_lj
from test_gpu_small import _random

pytestmark = pytest.mark.gpu

LJ, OP = (1.0, 1.0, 2.5, 2.5), (10000.0, 0.2, 100.0, 1.0)


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.mark.parametrize("L,n,model,params,applies", [
    ((5.3, 36.2, 31.1), 1500, "lj_shifted", LJ, 3),          # 2 x 14 x 12 spaces: rows listed as runs
    ((36.2, 31.1, 5.3), 1500, "lj_shifted", LJ, 3),          # two spaces along the rows
    ((10.3, 36.2, 25.6), 4000, "lj_shifted", LJ, 3),         # 4 x 14 x 10
    ((20.0, 20.0, 20.0), 700, "lj", (1.0, 1.0, 2.5), 3),     # spaces as wide as the cutoff: a scan of two
    ((60.3, 5.2), 90, "lj", (1.0, 1.0, 2.5), 6),             # 2D, 24 x 2
    ((60.3, 72.1), 2400, "lj_shifted", LJ, 4),               # 2D, 24 x 28
    ((36.2, 31.1, 35.3), 40, "lj", (1.0, 1.0, 2.5), 8),      # most spaces empty
    ((9.3, 12.2, 10.1), 1100, "overlap_penalty", OP, 6),     # a wavefront per trial
    ((25.3, 27.2, 26.1), 15000, "overlap_penalty", OP, 3),   # 16 lanes per trial, ragged regions
    ((210.3, 207.2), 30000, "overlap_penalty", OP, 2),       # 2D, 16 lanes
    ((51.3, 50.2, 49.1), 110000, "overlap_penalty", OP, 1),  # 8 lanes
    ((9.3, 12.2, 10.1), 1100, "overlap_penalty", (5.0, 0.9, 0.3, 1.0), 6),
])
def test_replays(hmc, L, n, model, params, applies):
    pos = _random(n, L, 7, 2.0 if model == "overlap_penalty" else 0.9)
    _replay_lj(hmc, np.array(L), pos, model, params, 1.2, 0.2, applies, seed=11)


def test_more_candidates_than_one_batch_of_loads(hmc):
    # 600 bodies in a few spaces of a box that is otherwise dilute
    rng = np.random.default_rng(5)
    L = np.array([36.2, 31.1, 35.3])
    pos = np.concatenate([_random(300, L, 3), rng.uniform(-3.0, 3.0, (600, 3))])
    _replay_lj(hmc, L, pos, "lj_shifted", LJ, 1.2, 0.1, 1, seed=2)


@pytest.mark.parametrize("L,n,model,params,regions", [
    ((36.2, 31.1, 35.3), 30000, "lj_shifted", LJ, True), ((60.3, 72.1), 2400, "lj_shifted", LJ, True),
    ((15.3, 17.2, 16.1), 4000, "overlap_penalty", OP, True), ((51.3, 50.2, 49.1), 110000, "overlap_penalty", OP, True),
    ((62.3, 63.2, 65.1), 240000, "overlap_penalty", OP, False)])
def test_both_forms_agree(hmc, L, n, model, params, regions):
    pos = _random(n, L, 9, 2.0 if model == "overlap_penalty" else 0.9)
    out = []
    for persistent in (True, False):
        sim = hmc.GpuParallelSweep(np.array(L), pos, model=model, params=params, persistent=persistent)
        counts = sim.run(0, 3, 1.2, 0.15, 4)
        assert (sim.stats()["regions"] > 0) == (regions and persistent)
        out.append((counts, np.concatenate([x.ravel() for x in sim.positions()]).view(np.uint64)))
        sim.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
