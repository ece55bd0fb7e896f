"""The lock between processes that persistent launches hold (csrc/turnstile.hpp): one
process at a time, in turn, given up with the process that holds it."""
import os
import pathlib
import subprocess
import sys
import textwrap
import time

import _pkg

ROOT = pathlib.Path(__file__).resolve().parent

WORKER = textwrap.dedent("""
    import os, sys, time
    sys.path.insert(0, sys.argv[1])
    import _pkg
    lib = _pkg.pkg().lib()
    path, key, rounds, log = sys.argv[2].encode(), int(sys.argv[3]), int(sys.argv[4]), sys.argv[5]
    assert lib.hmc_debug_turn(path, key, 0) == 1
    out = os.open(log, os.O_WRONLY | os.O_APPEND)
    os.write(out, b"ready\\n")
    while not os.path.exists(log + ".go"):
        time.sleep(0.001)
    for _ in range(rounds):
        assert lib.hmc_debug_turn(path, key, 1) == 1
        os.write(out, b"%d in\\n" % os.getpid())
        time.sleep(0.002)
        os.write(out, b"%d out\\n" % os.getpid())
        lib.hmc_debug_turn(path, key, 2)
    if len(sys.argv) > 6:
        lib.hmc_debug_turn(path, key, 1)
        os.write(out, b"%d in\\n" % os.getpid())
        time.sleep(60)
""")


def _start(tmp_path, key, rounds, *more):
    log = tmp_path / "log"
    log.touch()
    (tmp_path / "lock").touch()
    return subprocess.Popen([sys.executable, "-c", WORKER, str(ROOT), str(tmp_path / "lock"), str(key), str(rounds),
                             str(log), *more])


def _wait(cond, seconds=60.0):
    end = time.time() + seconds
    while not cond():
        assert time.time() < end
        time.sleep(0.002)


def test_one_at_a_time_and_in_turn(tmp_path):
    procs = [_start(tmp_path, 7, 40) for _ in range(3)]
    log = tmp_path / "log"
    _wait(lambda: log.read_text().count("ready") == 3)
    (tmp_path / "log.go").touch()
    assert [p.wait(60) for p in procs] == [0, 0, 0]
    lines = [x.split() for x in log.read_text().splitlines() if not x.startswith("ready")]
    assert len(lines) == 240
    for a, b in zip(lines[::2], lines[1::2]):
        assert a[0] == b[0] and (a[1], b[1]) == ("in", "out")
    # while all three want it nobody has it twice running (but for a queue not yet joined)
    turns = [a[0] for a in lines[::2]]
    last = min(len(turns) - 1 - turns[::-1].index(p) for p in set(turns))
    again = sum(x == y for x, y in zip(turns[:last], turns[1:last]))
    assert again <= 6


def test_keys_do_not_meet(tmp_path):
    lib = _pkg.pkg().lib()
    (tmp_path / "lock").touch()
    assert lib.hmc_debug_turn(str(tmp_path / "lock").encode(), 3, 0) == 1
    assert lib.hmc_debug_turn(b"", 3, 1) == 1
    p = _start(tmp_path, 4, 5)
    (tmp_path / "log.go").touch()
    assert p.wait(60) == 0
    assert lib.hmc_debug_turn(b"", 3, 3) == 0
    lib.hmc_debug_turn(b"", 3, 2)


def test_a_waiting_process_is_seen_and_a_dead_one_gives_up(tmp_path):
    lib = _pkg.pkg().lib()
    p = _start(tmp_path, 9, 0, "hold")
    (tmp_path / "log.go").touch()
    _wait(lambda: " in" in (tmp_path / "log").read_text())
    path = str(tmp_path / "lock").encode()
    assert lib.hmc_debug_turn(path, 9, 0) == 1
    p.kill()
    p.wait()
    assert lib.hmc_debug_turn(path, 9, 1) == 1  # (waits for the other's end at most)
    q = _start(tmp_path, 9, 1)
    _wait(lambda: lib.hmc_debug_turn(path, 9, 3) == 1)
    lib.hmc_debug_turn(path, 9, 2)
    assert q.wait(60) == 0


def test_no_file_no_lock(tmp_path):
    lib = _pkg.pkg().lib()
    assert lib.hmc_debug_turn(str(tmp_path / "none").encode(), 1, 0) == 0
