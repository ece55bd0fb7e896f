"""The waits and reloads of a persistent apply's regions, played through on the CPU with
the library's own rules: regions start and end their passes in random order, as far as
their waits let them, and at every moment a region in a pass must find the halo cells
that the pass reads neither being written nor older or newer than the pass before,
in the sites of the neighbours and in its own copy."""
import ctypes as C
import functools
import itertools
import random

import pytest

import _pkg


def _rule(dim, kind, a, rl=None):
    v = (C.c_int32 * 3)(*a)
    r = None if rl is None else (C.c_int32 * 3)(*rl)
    return _pkg.pkg().lib().hmc_debug_region_rule(dim, kind, v, r)


@functools.lru_cache(None)
def _distance(dim, j, axes):
    return _rule(dim, 0, (j, axes))


@functools.lru_cache(None)
def _halo(dim, T, rl):
    """(local cell, axes it lies in the halo of, colour, reload pass) of a region's box."""
    out = []
    for lc in itertools.product(*[range(-1, 2 * T[a] + 1) for a in range(dim)]):
        q = _rule(dim, 1, lc, rl)
        axes = sum(1 << (dim - 1 - a) for a in range(dim) if lc[a] < 0 or lc[a] == rl[a])
        inside = all(lc[a] <= rl[a] for a in range(dim))
        assert (q == 0xFFFFFFFF) == (not inside or not axes)
        if inside and axes:
            out.append((lc, axes, sum(1 << (dim - 1 - a) for a in range(dim) if lc[a] & 1), q))
    return out


def _play(dim, shape, T, passes, seed):
    rnd, colours = random.Random(seed), 1 << dim
    nt = [-(-(shape[a] // 2) // T[a]) for a in range(dim)]
    regions = list(itertools.product(*[range(n) for n in nt]))
    rl = {t: tuple(min(2 * T[a], shape[a] - 2 * T[a] * t[a]) for a in range(dim)) for t in regions}
    owner = {tuple(2 * T[a] * t[a] + o[a] for a in range(dim)): t
             for t in regions for o in itertools.product(*[range(rl[t][a]) for a in range(dim)])}
    halo = {}
    for t in regions:
        cells = [(lc, owner[tuple((2 * T[a] * t[a] + lc[a]) % shape[a] for a in range(dim))], axes, k, q)
                 for lc, axes, k, q in _halo(dim, T, rl[t])]
        halo[t] = [c for c in cells if c[1] != t]
    done, started, copy = dict.fromkeys(regions, 0), dict.fromkeys(regions, 0), {}
    bias = {t: 0.95 * rnd.random() ** 3 for t in regions}

    def version(passes_of, k):  # how often colour k of a region has been written
        return passes_of // colours + (passes_of % colours > k)

    def neighbour(t, axes, j):  # on the sides that pass j reads
        return tuple((t[a] + (0 if not axes >> (dim - 1 - a) & 1 else 1 if j >> (dim - 1 - a) & 1 else -1)) % nt[a]
                     for a in range(dim))

    def check(t):
        j = started[t] - 1
        for lc, y, axes, k, _ in halo[t]:
            # colour bit 0 reads the lower side, 1 the upper one
            if any(axes >> (dim - 1 - a) & 1 and (lc[a] < 0) == bool(j >> (dim - 1 - a) & 1) for a in range(dim)):
                continue
            want = version(j, k)
            assert version(done[y], k) == version(started[y], k) == want, (t, j, lc)
            assert copy[t][lc] == want, (t, j, lc)

    while min(done.values()) < passes:
        for t in rnd.sample(regions, len(regions)):
            if done[t] >= passes or rnd.random() < bias[t]:
                continue
            if started[t] > done[t]:
                check(t)
                done[t] += 1
            elif t not in copy:  # staged late, while neighbours write
                copy[t] = {lc: version(rnd.choice((done, started))[y], k) for lc, y, _, k, _ in halo[t]}
            else:
                j = done[t]
                waits = [(neighbour(t, axes, j), j - _distance(dim, j, axes) + 1) for axes in range(1, colours)]
                if any(need > 0 and n != t and done[n] < need for n, need in waits):
                    continue
                if j:
                    copy[t].update({lc: version(done[y], k) for lc, y, _, k, q in halo[t] if q == j % colours})
                started[t] += 1
                for u in regions:
                    if started[u] > done[u]:
                        check(u)
    return nt


@pytest.mark.parametrize("seed", range(3))
def test_plane(seed):
    seen = set()
    for T in itertools.product((1, 2, 3), repeat=2):
        for shape in itertools.product((6, 8, 10, 12), repeat=2):
            if all(2 * T[a] + 2 <= shape[a] - 2 for a in range(2)):
                nt = [-(-(shape[a] // 2) // T[a]) for a in range(2)]
                if max(nt) <= 4 and (T, shape) not in seen:
                    seen.add((T, shape))
                    _play(2, shape, T, 12, seed)
    assert len(seen) > 30


@pytest.mark.parametrize("seed", range(2))
@pytest.mark.parametrize("shape,T", [((6, 6, 6), (1, 1, 1)), ((8, 10, 12), (2, 3, 2)), ((6, 6, 10), (1, 1, 3)),
                                     ((12, 10, 14), (2, 2, 2)), ((8, 8, 8), (2, 1, 2)), ((6, 12, 8), (1, 2, 2))])
def test_space(shape, T, seed):
    _play(3, shape, T, 20, seed)
