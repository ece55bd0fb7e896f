"""The persistent applies at the edges of what their regions and fast paths
take: the fewest spaces per axis, ragged last regions, rows of more sites than
the unrolled walk reads on past, sites without images, coordinates of exactly
zero, and the division by a constant behind the wrapped positions.  Replays
are compared with the oracle bit for bit (trace, counts, positions)."""
import sys

import numpy as np
import pytest

import _pkg
from test_gpu_parity import _replay

pytestmark = pytest.mark.gpu


def log(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.fixture(scope="module")
def wl():
    return _pkg.workloads()


@pytest.mark.parametrize("b", [6.448, 10.0 / 3.0, 101.56, 1.0078125, 3.0, np.nextafter(4.0, 0.0), np.nextafter(1.0, 2.0),
                               1e30, 1e-30, 2.0**120])
def test_division_by_a_constant_is_ieee(hmc, b):
    # quotients of every exponent the fast form takes and of the two beside it,
    # significands at both ends, and the range positions have
    rng = np.random.default_rng(17)
    n = 1 << 18
    a = np.concatenate([rng.uniform(-1.0, 1.0, n) * b, rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-901, 902, n),
                        (1.0 + 2.0**-52 * rng.integers(0, 64, n)) * 2.0 ** rng.integers(-2, 8, n),
                        (2.0 - 2.0**-52 * rng.integers(1, 64, n)) * 2.0 ** rng.integers(-2, 8, n),
                        [0.0, b, -b, b / 2, 1e-310, 2.0**-900, 2.0**900]])
    x = np.stack([a, np.full_like(a, b)], 1)
    assert np.array_equal(hmc.debug_math("div_const", x.ravel()), a / b)


@pytest.mark.parametrize("cells,phi,d", [((4, 4, 4), 0.50, 0.08), ((5, 9, 13), 0.42, 0.15), ((17, 4, 6), 0.50, 0.08),
                                         ((11, 12, 7), 0.54, 0.05), ((8, 8, 8), 0.05, 0.9)])
def test_region_shapes_3d(hmc, wl, cells, phi, d):
    L, pos = wl.fcc_spheres(cells, packing_fraction=phi)
    st = _replay(hmc, L, pos, d, 8, "mixed")
    assert st["tiled"] == 2
    log(f"{cells} phi {phi}: {st['regions']} regions of {st['tile_shape']}")


@pytest.mark.parametrize("nx,ny,phi", [(7, 7, 0.70), (9, 41, 0.60), (64, 7, 0.72), (33, 29, 0.05)])
def test_region_shapes_2d(hmc, wl, nx, ny, phi):
    a = np.sqrt(np.pi / 4.0 / phi)
    L = np.array([nx * a, ny * a])
    i, j = np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij")
    pos = np.stack([(i.ravel() + 0.5) * a, (j.ravel() + 0.5) * a], 1) - L / 2
    st = _replay(hmc, L, pos, 0.15, 12, "mixed")
    assert st["tiled"] == 2


def test_rows_longer_than_the_walk_reads_past(hmc, wl):
    # 24 overlapping bodies in one space of a dilute box that still fits the
    # regions' capacity: its rows are walked one site at a time
    L, pos = wl.fcc_spheres((6, 6, 6), packing_fraction=0.30)
    rng = np.random.default_rng(2)
    pos = np.concatenate([pos, rng.uniform(0.05, 0.45, (24, 3))])
    st = _replay(hmc, L, pos, 0.3, 10, "mixed", seed=9)
    assert st["tiled"] == 2 and st["tile_overflows"] == 0


def test_sites_without_images(hmc, wl):
    # given sites at L/2 exactly (a wrapped one never is) have no ghosts in the
    # reference; their entries are NaN and every pair with them is re-tested:
    # the same run as the trials from global memory in FP64
    L = np.array([10.5, 9.3, 9.6])  # spaces wider than the diameter on every axis
    rng = np.random.default_rng(5)
    pos = wl.random_dilute(150, L, 3, 1.0, seed=4)
    edge = np.stack([np.full(12, np.nextafter(5.25, 0.0)), rng.uniform(-4.4, 4.4, 12), rng.uniform(-4.6, 4.6, 12)], 1)
    body = wl.wrap(L, np.concatenate([pos, edge]))
    site = body.copy()
    site[150:, 0] = 5.25
    out = []
    for kw in (dict(precision="mixed"), dict(precision="fp64", lds_tiles=False)):
        sim = hmc.GpuParallelSweep(L, body, sites=site, **kw)
        cnt = [sim.run(k, 3, 1.0, 0.2, 1) for k in range(10)]
        out.append((cnt, *sim.positions()))
        assert sim.stats()["tiled"] == (2 if kw["precision"] == "mixed" else 0)
        sim.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])


def test_coordinates_of_exactly_zero(hmc, wl):
    # positions on the planes through the origin, and moves far below the ulp of
    # the others: the proposal's general form
    L, pos = wl.fcc_spheres((5, 5, 5), packing_fraction=0.45)
    pos = pos - pos[137]
    st = _replay(hmc, L, pos, 1e-300, 3, "mixed")
    assert st["tiled"] == 2
    _replay(hmc, L, pos, 0.1, 6, "mixed")


@pytest.mark.parametrize("cells,phi,d", [((4, 4, 4), 0.50, 0.08), ((5, 9, 13), 0.42, 0.15), ((29, 23, 31), 0.45, 0.1),
                                         ((8, 8, 8), 0.05, 0.9)])
def test_fp64_regions(hmc, wl, cells, phi, d):
    # FP64 box-relative entries with the exact re-test inside the band
    L, pos = wl.fcc_spheres(cells, packing_fraction=phi)
    st = _replay(hmc, L, pos, d, 6, "fp64")
    assert st["tiled"] == 1 and st["regions"] > 0
    log(f"{cells} phi {phi}: {st['regions']} regions of {st['tile_shape']}, {st['band_retests']} re-tests")
