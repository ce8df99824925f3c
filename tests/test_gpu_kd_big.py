"""kd orders of candidate sets beyond 8,192 entries, each alone (the launches of
one molecule) and together: coordinates as in PDB files (many equal ones),
without any equal ones, with a single equal pair across the root's split
point, and in order. The orders must be the oracle's QuickSelect orders, element
for element."""

import time

import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


def points(style, n):
    rng = np.random.default_rng([n, len(style)])
    xyz = rng.normal(size=(n, 3)) * 20.0
    if style == "pdb":
        return np.round(xyz, 3)
    if style == "one tie":
        x = np.sort(xyz[:, 0])
        i, j = np.flatnonzero(xyz[:, 0] == x[n // 2 - 1])[0], np.flatnonzero(xyz[:, 0] == x[n // 2])[0]
        xyz[j, 0] = xyz[i, 0]
    if style == "sorted":
        x = np.arange(n, dtype=np.float64)
        xyz = np.stack([x, -x, np.zeros(n)], axis=1)
    return xyz


def want_of(xyz):
    n = len(xyz)
    blank = np.full((n, 4), ord("_"), np.uint8)
    mol = oracle.MolView(xyz, blank, blank, np.zeros(n, np.uint8), np.zeros(n, np.int32), np.arange(n, dtype=np.int32))
    return oracle.kd_order(mol, np.arange(n, dtype=np.int32))


@pytest.mark.parametrize("style", ["pdb", "free", "one tie", "sorted"])
def test_orders(style):
    from pyjess_amd import _native

    sizes = [8193, 9000, 16384, 16385, 20001]
    sets = [points(style, n) for n in sizes]
    want = [want_of(p) for p in sets]
    for p, w in zip(sets, want):
        print(style, len(p), flush=True)
        assert _native.kd_order(p, np.array([0, len(p)])).tolist() == w
    off = np.concatenate([[0], np.cumsum(sizes)])
    got = _native.kd_order(np.concatenate(sets), off)
    for k, w in enumerate(want):
        assert got[off[k]:off[k + 1]].tolist() == w


def test_fast_path_of_one_molecule():
    """Without equal coordinates a large set takes no longer alone than as one of
    two (which run beside each other, by the fast path)."""
    from pyjess_amd import _native

    xyz = points("free", 100000)

    def least(sets):
        off = len(xyz) * np.arange(sets + 1)
        times = []
        for _ in range(4):
            t0 = time.perf_counter()
            _native.kd_order(np.tile(xyz, (sets, 1)), off)
            times.append(time.perf_counter() - t0)
        return min(times)

    one, two = least(1), least(2)
    print(one, two, flush=True)
    assert one < 1.2 * two
