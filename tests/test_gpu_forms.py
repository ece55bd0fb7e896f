"""Which kernels a context's applies take: the rules' lines, from both sides."""
import numpy as np
import pytest

import _pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def _lattice(L, n, seed=1, jitter=0.02):
    # n sites of a cubic or square lattice that fills the box, slightly displaced
    L = np.asarray(L, float)
    d = len(L)
    m = np.maximum(1, np.ceil((n / np.prod(L)) ** (1.0 / d) * L).astype(int))
    g = np.stack(np.meshgrid(*[np.arange(k) for k in m], indexing="ij"), -1).reshape(-1, d)
    rng = np.random.default_rng(seed)
    g = g[np.sort(rng.permutation(len(g))[:n])]
    return (g + 0.5) * (L / m) - L / 2 + rng.uniform(-jitter, jitter, (len(g), d)) * (L / m)


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("L,n,width,bucket", [
    ((25.3, 26.3, 27.3), 9000, 1.0, True), ((25.0, 26.0, 27.0), 9000, 1.55, True),
    ((25.0, 26.0, 27.0), 9000, 1.75, False), ((25.0, 26.0, 27.0), 9000, 2.4, False),
    ((25.0, 26.0, 27.0), 900, 2.4, False), ((61.0, 62.0), 2300, 2.0, True), ((61.0, 62.0), 2300, 4.0, False)])
def test_build_of_wide_spaces(hmc, L, n, width, bucket, precision):
    # a body interaction range beyond the diameter: spaces of many bodies, which
    # the buckets of the two-kernel build do not hold
    L, pos = np.array(L), _lattice(L, n)
    out = []
    for persistent in (True, False):
        sim = hmc.GpuParallelSweep(L, pos, precision=precision, body_interaction_range=width, persistent=persistent)
        form = sim.debug_form()
        assert form["persistent"] == int(persistent) and form["bucket_build"] == int(bucket and persistent)
        counts = sim.run(0, 3, 1.0, 0.15, 2)
        out.append((counts, np.concatenate([x.ravel() for x in sim.positions()]).view(np.uint64)))
        sim.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("L,n,model,form", [
    ((120.0, 121.0), 10000, "lj_shifted", dict(persistent=0, iso_lanes=64)),  # a scan of two, 576 trials a colour
    ((375.0, 376.0), 100000, "lj_shifted", dict(persistent=0, iso_lanes=8)),  # 5,625
    ((250.0, 251.0), 10000, "lj_shifted", dict(persistent=0, iso_lanes=8)),  # 2,500, nine candidates
    ((20.0, 21.3, 22.3), 9000, "overlap_penalty", dict(persistent=0, iso_lanes=64)),  # 1,100
    ((32.0, 33.3, 34.3), 33000, "overlap_penalty", dict(persistent=0, iso_lanes=8)),  # 4,352
    ((60.3, 72.1), 2400, "lj_shifted", dict(persistent=1, iso_lanes=64)),
    ((25.3, 27.2, 26.1), 15000, "overlap_penalty", dict(persistent=1, iso_lanes=16)),
    ((51.3, 50.2, 49.1), 110000, "overlap_penalty", dict(persistent=1, iso_lanes=8)),
    ((36.2, 31.1, 35.3), 30000, "lj_shifted", dict(persistent=1, iso_lanes=64)),
    ((9.3, 12.2, 10.1), 1100, "overlap_penalty", dict(persistent=1, iso_lanes=64, small_waves=0)),
    ((15.5, 15.4, 15.3), 1100, "lj_shifted", dict(persistent=0, iso_lanes=0, small_waves=1)),
    ((10.1, 10.2, 10.3), 700, "lj_shifted", dict(persistent=0, iso_lanes=0, small_waves=2)),
    ((5.3, 5.2, 5.4), 60, "lj_shifted", dict(persistent=0, iso_lanes=0, small_waves=4)),
])
def test_lanes_of_pair_energies(hmc, L, n, model, form):
    sim = hmc.GpuParallelSweep(np.array(L), _lattice(L, n), model=model)
    got = sim.debug_form()
    sim.close()
    assert {k: got[k] for k in form} == form
