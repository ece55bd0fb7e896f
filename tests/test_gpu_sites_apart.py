"""Given sites that lie away from their bodies: a trial still meets the sites of all
bodies in the spaces around its own, in every form of an apply.  The per-colour hard-shape
and mixed-precision LJ passes, which visit every neighbour space, are the reference."""
import numpy as np
import pytest

import _oracle as O
import _pkg
from test_gpu_forms import _lattice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


def _wrap(L, x):
    return O.wrap(L, np.ascontiguousarray(x))


def _pairs(rng, L, gap, away):
    """Bodies X on a sparse lattice and, for each, a body Y in a space next to its
    space on the diagonal, whose site lies on X's."""
    k = np.floor(np.asarray(L) / gap).astype(int)
    g = np.stack(np.meshgrid(*[np.arange(n) for n in k], indexing="ij"), -1).reshape(-1, len(L))
    x = (g + 0.5) * (np.asarray(L) / k) - np.asarray(L) / 2 + rng.uniform(-0.3, 0.3, g.shape)
    y = x + away * rng.choice([-1.0, 1.0], x.shape)
    x, y = _wrap(L, x), _wrap(L, y)
    return np.concatenate([x, y]), np.concatenate([x, _wrap(L, x + rng.uniform(-0.02, 0.02, x.shape))])


def _run(sim, d, kT=1.0, n=3):
    out = []
    for k in range(n):
        out.append(sim.apply(k, 0, 9, kT, d))
    res = out, [p.view(np.uint64) for p in sim.positions()]
    return res


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("L", [(25.2, 26.2, 27.3), (61.2, 62.3)])
def test_hard_shapes(hmc, L, precision):
    L = np.array(L)
    body, site = _pairs(np.random.default_rng(3), L, 3.6, 0.9)
    out = []
    for kw in (dict(), dict(persistent=False), dict(lds_tiles=False)):
        sim = hmc.GpuParallelSweep(L, body, sites=site, precision=precision, **kw)
        out.append(_run(sim, 0.1))
        sim.close()
    for o in out[1:]:
        assert out[0][0] == o[0] and all(np.array_equal(a, b) for a, b in zip(out[0][1], o[1]))
    # bodies with their own sites take the persistent form again
    sim = hmc.GpuParallelSweep(L, body, sites=site, precision=precision)
    forms = [sim.debug_form()["persistent"]]
    sim.set_positions(body)
    forms.append(sim.debug_form()["persistent"])
    sim.set_positions(*sim.positions())
    forms.append(sim.debug_form()["persistent"])
    sim.close()
    assert forms == [0, 1, 1]


@pytest.mark.parametrize("L,rc", [((31.0, 32.3, 33.1), 2.5), ((15.3, 16.1, 15.9), 2.5), ((9.3, 10.2, 12.1), 2.5),
                                  ((61.0, 62.3), 2.5), ((20.0, 20.0, 20.0), 2.5)])
def test_lennard_jones(hmc, L, rc):
    # persistent launches of 64 lanes, one workgroup, 2D, a scan of two; mixed
    # precision per colour decides every trial as FP64 does
    L, rng = np.array(L), np.random.default_rng(4)
    body = _lattice(L, int(0.3 * np.prod(L)) if len(L) == 3 else 1500, jitter=0.1)
    site = _wrap(L, body + rng.uniform(-1.2, 1.2, body.shape))
    out = []
    for kw in (dict(), dict(persistent=False), dict(precision="mixed"), dict(precision="mixed", persistent=False)):
        sim = hmc.GpuParallelSweep(L, body, sites=site, model="lj_shifted", params=(1.0, 1.0, rc, rc), **kw)
        out.append(_run(sim, 0.3, kT=2.0, n=2))
        assert sim.stats()["ambiguous"] == 0
        sim.close()
    for o in out[:-1]:
        assert out[-1][0] == o[0] and all(np.array_equal(a, b) for a, b in zip(out[-1][1], o[1]))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("persistent", [True, False])
def test_convex(hmc, precision, persistent):
    # a trial of X overlaps Y's site until Y has moved and taken its site along
    cube = np.array([[a, b, c] for a in (-0.5, 0.5) for b in (-0.5, 0.5) for c in (-0.5, 0.5)])
    tried = 0
    for seed in range(4):
        L = np.array([29.0, 30.1, 31.2])
        body, site = _pairs(np.random.default_rng(seed), L, 5.0, 1.55)
        n = len(body) // 2
        sim = hmc.GpuParallelSweep(L, body, sites=site, model="convex", vertices=cube, precision=precision,
                                   persistent=persistent)
        sim.trace(True, capacity=1 << 16)
        sim.apply(0, 0, seed, 1.0, 0.1)
        t = sim.read_trace(capacity=1 << 16)
        sim.close()
        t = t[np.lexsort((t["color"], t["substep"]))]
        moved = set()
        for r in t:
            b = int(r["body"])
            if b < n and b + n not in moved:
                tried += 1
                assert r["status"] != 1, (seed, b)
            if r["status"] == 1:
                moved.add(b)
    assert tried > 100


def test_scale_distribution_function(hmc):
    # all sites shifted alike: neighbours within r_max are still bodies of spaces
    # next to one another
    for L in (np.array([12.0, 13.0, 14.0]), np.array([30.0, 31.0])):
        body = _lattice(L, int(0.5 * np.prod(L)), jitter=0.2)
        site = _wrap(L, body + np.array([0.45, -0.4, 0.35])[: len(L)])
        want, wov = O.sdf(L, site, 1.0, 0.1, 0.001, 100, all_pairs=True)
        sim = hmc.GpuParallelSweep(L, body, sites=site)
        h, ov = sim.sdf(0.1, 0.001, nbins=100)
        sim.close()
        assert np.array_equal(h, want) and ov == wov
        batch = hmc.GpuBatch([(L, body, None), (L, body, site)])
        h, ov = batch.sdf(0.1, 0.001, nbins=100)
        batch.close()
        want0, _ = O.sdf(L, _wrap(L, body), 1.0, 0.1, 0.001, 100, all_pairs=True)
        assert np.array_equal(h[1], want) and ov[1] == wov and np.array_equal(h[0], want0)


def test_batch(hmc):
    systems = []
    for r in range(6):
        L = np.array([14.2 + r, 15.2, 16.3])
        body, site = _pairs(np.random.default_rng(r), L, 3.6, 0.9)
        systems.append((L, body, site if r % 2 else None))
    out = []
    for persistent in (True, False):
        b = hmc.GpuBatch(systems, precision="mixed", persistent=persistent)
        cnt = b.run(0, np.arange(6), 1.0, 0.1, 3)
        forms = [b.stats(0)["tiled"]]
        pos = [b.positions(r) for r in range(6)]
        for r in range(6):
            b.set_positions(r, systems[r][1])
        b.run(3, np.arange(6), 1.0, 0.1, 1)
        forms.append(b.stats(0)["tiled"])
        out.append((cnt, np.concatenate([p.ravel() for q in pos for p in q]).view(np.uint64), forms))
        b.close()
    assert np.array_equal(np.asarray(out[0][0]), np.asarray(out[1][0])) and np.array_equal(out[0][1], out[1][1])
    assert out[0][2] == [1, 2] and out[1][2] == [1, 1]
