"""Two processes with persistent applies on one device: each ends where it does alone,
and none waits for the other's whole run."""
import pathlib
import subprocess
import sys
import textwrap
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = pathlib.Path(__file__).resolve().parent

WORKER = textwrap.dedent("""
    import os, sys, time
    sys.path.insert(0, sys.argv[1])
    import numpy as np
    import _pkg
    hmc, wl = _pkg.pkg(), _pkg.workloads()
    kind, out, steps, calls = sys.argv[2], sys.argv[3], int(sys.argv[4]), int(sys.argv[5])
    if kind == "spheres":
        L, p = wl.fcc_spheres((30, 30, 30), packing_fraction=0.5)
        sim = hmc.GpuParallelSweep(L, wl.wrap(L, p), precision="mixed")
    else:
        L, p = wl.fcc_spheres((20, 20, 20), packing_fraction=0.45)
        sim = hmc.GpuParallelSweep(L, wl.wrap(L, p), model="overlap_penalty")
    assert sim.debug_form()["persistent"] == 1
    sim.run(0, 5, 1.0, 0.08, 2)
    open(out + ".ready", "w").close()
    while not os.path.exists(sys.argv[6]):
        time.sleep(0.001)
    ends = []
    for k in range(calls):
        sim.run(2 + steps * k, 5, 1.0, 0.08, steps)
        ends.append(time.time())
    np.savez(out, pos=sim.positions()[0], ends=np.array(ends), start=os.path.getmtime(sys.argv[6]))
    sim.close()
""")


def _run(tmp_path, jobs):
    go = tmp_path / "go"
    if go.exists():
        go.unlink()
    procs, outs = [], []
    for i, (kind, steps, calls) in enumerate(jobs):
        out = tmp_path / f"{kind}{i}.npz"
        ready = pathlib.Path(str(out) + ".ready")
        if ready.exists():
            ready.unlink()
        outs.append(out)
        procs.append(subprocess.Popen([sys.executable, "-c", WORKER, str(ROOT), kind, str(out), str(steps), str(calls),
                                       str(go)]))
    end = time.time() + 60
    while not all(pathlib.Path(str(o) + ".ready").exists() for o in outs):
        assert time.time() < end and all(p.poll() is None for p in procs)
        time.sleep(0.01)
    go.touch()
    assert [p.wait(60) for p in procs] == [0] * len(procs)
    return [np.load(o) for o in outs]


def test_two_processes(tmp_path):
    jobs = [("spheres", 40, 20), ("penalty", 2000, 1)]
    alone = [_run(tmp_path, [j])[0]["pos"].copy() for j in jobs]
    both = _run(tmp_path, jobs)
    for a, b in zip(alone, both):
        assert np.array_equal(a.view(np.uint64), b["pos"].view(np.uint64))
    # the short calls of the first end while the one long call of the second runs
    assert both[0]["ends"][0] < both[1]["ends"][-1]
