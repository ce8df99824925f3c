"""Exact kd pass on the device at the edges of its launch shapes: one wave
(64 positions), one, two, four and eight positions per thread, the windows
that pass from the workgroup to one wave (64/65 positions) and sets beside
larger and smaller ones of other tiers, alone and in batches. The leaf orders
must be the oracle's QuickSelect orders, element for element."""

import numpy as np
import pytest

SIZES = [1, 2, 3, 63, 64, 65, 127, 128, 129, 130, 191, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048,
         2049, 4095, 4096, 4097, 8191, 8192]


def points(style, n, seed):
    rng = np.random.default_rng([seed, n])
    if style == "grid":        # many equal coordinates
        return rng.integers(0, 6, size=(n, 3)).astype(np.float64)
    if style == "sorted":      # one long run of "<=" or ">" keys per partition
        x = np.arange(n, dtype=np.float64)
        return np.stack([x, -x, np.zeros(n)], axis=1)
    return np.round(rng.normal(size=(n, 3)) * 20.0, 3)


def test_hop_quotient_is_exact():
    """floor((run + 0.5) / s) in float, with a reciprocal up to two ulp off,
    is run // s for every run inside a 64-bit word."""
    s = np.arange(1, 8193, dtype=np.int64)[:, None]
    run = np.arange(64, dtype=np.int64)[None, :]
    rcp = (np.float32(1.0) / s.astype(np.float32)).astype(np.float32)
    for ulps in (-2, -1, 0, 1, 2):
        r = (rcp.view(np.int32) + np.int32(ulps)).view(np.float32)
        assert np.array_equal(((run.astype(np.float32) + np.float32(0.5)) * r).astype(np.int64), run // s)


@pytest.mark.gpu
@pytest.mark.parametrize("style", ["pdb", "grid", "sorted"])
def test_exact_pass_at_tile_edges(style):
    from oracle import oracle
    from pyjess_amd import _native

    def want_of(xyz):
        n = len(xyz)
        blank = np.full((n, 4), ord("_"), np.uint8)
        mol = oracle.MolView(xyz, blank, blank, np.zeros(n, np.uint8), np.zeros(n, np.int32),
                             np.arange(n, dtype=np.int32))
        return oracle.kd_order(mol, np.arange(n, dtype=np.int32))

    sets = [points(style, n, 5) for n in SIZES]
    want = [want_of(p) for p in sets]
    # each alone (the launches of one molecule), then all in one batch
    for p, w in zip(sets, want):
        print(style, len(p), "alone", flush=True)
        assert _native.kd_order(p, np.array([0, len(p)])).tolist() == w, (style, len(p))
    off = np.concatenate([[0], np.cumsum(SIZES)])
    got = _native.kd_order(np.concatenate(sets), off)
    for k, w in enumerate(want):
        assert got[off[k]:off[k + 1]].tolist() == w, (style, SIZES[k])
