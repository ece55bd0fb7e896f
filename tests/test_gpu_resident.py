"""Persistent applies of several contexts on one device: interleaved from one
thread, from a thread each at the same time, and with contexts made and closed in
between.  Every context ends where it does alone."""
import threading

import numpy as np
import pytest

import _pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmc():
    p = _pkg.pkg()
    p.lib()
    return p


@pytest.fixture(scope="module")
def wl():
    return _pkg.workloads()


def _make(hmc, wl, k):
    if k == 0:
        L, p = wl.fcc_spheres((30, 30, 30), packing_fraction=0.5)
        return hmc.GpuParallelSweep(L, wl.wrap(L, p), precision="mixed")
    if k == 1:
        L, p = wl.fcc_number_density((12, 12, 12), 0.8)
        return hmc.GpuParallelSweep(L, wl.wrap(L, p), model="lj_shifted", params=(1.0, 1.0, 2.5, 2.5), precision="mixed")
    if k == 2:
        L, p = wl.fcc_spheres((20, 20, 20), packing_fraction=0.45)
        return hmc.GpuParallelSweep(L, wl.wrap(L, p), model="overlap_penalty")
    systems = [(L, p, None) for L, p in wl.batched_replicas(6, k_range=(6, 14), phi_range=(0.3, 0.5))]
    return hmc.GpuBatch(systems, precision="mixed")


def _run(sim, step, n):
    if hasattr(sim, "R"):
        sim.run(step, np.arange(sim.R), 1.0, 0.08, n)
    else:
        sim.run(step, 5, 1.0, 0.08, n)


def _state(sim):
    if hasattr(sim, "R"):
        return np.concatenate([sim.positions(r)[0].ravel() for r in range(sim.R)]).view(np.uint64)
    return sim.positions()[0].ravel().view(np.uint64)


@pytest.fixture(scope="module")
def alone(hmc, wl):
    out = []
    for k in range(4):
        sim = _make(hmc, wl, k)
        for i in range(6):
            _run(sim, 4 * i, 4)
        out.append(_state(sim))
        sim.close()
    return out


def test_interleaved(hmc, wl, alone):
    sims = [_make(hmc, wl, k) for k in range(4)]
    for i in range(6):
        for sim in sims:
            _run(sim, 4 * i, 4)
        extra = _make(hmc, wl, i % 4)
        _run(extra, 0, 1)
        extra.close()
    for sim, want in zip(sims, alone):
        assert np.array_equal(_state(sim), want)
        sim.close()


def test_a_thread_each(hmc, wl, alone):
    got, errors = [None] * 4, []

    def work(k):
        try:
            sim = _make(hmc, wl, k)
            for i in range(6):
                _run(sim, 4 * i, 4)
            got[k] = _state(sim)
            sim.close()
        except Exception as e:  # noqa: BLE001 (reported by the main thread)
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for g, want in zip(got, alone):
        assert np.array_equal(g, want)
