"""Point sets larger than the RMSD kernels hold in LDS: sets of 383 to 385 points
(half a buffer and one point to either side), 769 and 1,000 among small ones; tiles of
many sets that take rounds, chunks of points, or both arrays from global
memory. Few sets and the same sets among many (the kernels' two forms, which
do the same operations in the same order) must agree bit for bit."""

import numpy as np
import pytest

from oracle.kabsch_torch import kabsch_rmsd_grad
from tests.test_gpu_autograd import device, pairs, run
from tests.test_rmsd_grad_cpu import exact_rmsd

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TILES = {
    "large among small": [3, 383, 5, 384, 7, 385, 1, 769, 4, 1000, 6, 2],
    "rounds": [13, 20, 16, 24, 12],
    "one above 12": [3, 5, 11, 4, 8, 30, 2, 12],
    "chunks": [40, 1, 33, 64, 50],
    "multiples of a chunk": [35, 36, 34, 40, 45],
    "all large": [130, 129, 128, 127],
}


def sets_of(sizes, n_sets, seed):
    k = np.array([sizes[s % len(sizes)] for s in range(n_sets)])
    a, b, _ = pairs(n_sets, seed, k_min=int(k.max()), k_max=int(k.max()), collinear=0.0)
    keep = np.concatenate([np.arange(x) + s * int(k.max()) for s, x in enumerate(k)])
    return a[keep], b[keep], np.concatenate([[0], np.cumsum(k)]).astype(np.int64)


@pytest.mark.parametrize("kind", list(TILES))
@pytest.mark.parametrize("n_sets", [12, 64, 70])
def test_values_and_forms(kind, n_sets):
    print(kind, n_sets, flush=True)
    a, b, off = sets_of(TILES[kind], n_sets, 17)
    w = np.random.default_rng(3).uniform(-1.0, 1.0, size=n_sets)
    r, ga, gb = run(a, b, off, weights=w)
    for s in range(0, n_sets, 1 + n_sets // 12):
        A, B = a[off[s]:off[s + 1]], b[off[s]:off[s + 1]]
        want = exact_rmsd(A, B)
        # n additions, each rounded once, against the 50-digit value
        assert abs(r[s] - want) <= max(1e-13, len(A) * 2.0 ** -52) * max(1.0, want), s
        if len(A) < 4:
            continue   # (nearly) flat: the gradient of the reference loses digits
        _, ta, tb = kabsch_rmsd_grad(A, B)
        x = np.concatenate([ga[off[s]:off[s + 1]], gb[off[s]:off[s + 1]]]).ravel()
        y = w[s] * np.concatenate([ta, tb]).ravel()
        assert np.linalg.norm(x - y) <= 1e-10 * np.linalg.norm(y), s
    # the same sets at the head of more than 65,536
    rest = 65600
    tail = pairs(1, 5, k_min=2, k_max=2, collinear=0.0)
    a2, b2 = (np.concatenate([x, np.tile(t, (rest, 1))]) for x, t in ((a, tail[0]), (b, tail[1])))
    off2 = np.concatenate([off, off[-1] + 2 * np.arange(1, rest + 1)])
    r2, ga2, gb2 = run(a2, b2, off2, weights=np.concatenate([w, np.ones(rest)]))
    assert np.array_equal(r2[:n_sets], r)
    assert np.array_equal(ga2[:off[-1]], ga) and np.array_equal(gb2[:off[-1]], gb)
    assert np.all(r2[n_sets:] == r2[n_sets])


def elapsed(n_sets, k):
    """Device time of forward and backward over sets of k points (the least of a
    few runs), in ms."""
    from pyjess_amd.autograd import superposition_rmsd

    g = torch.Generator(device=device()).manual_seed(1)
    a, b = (torch.randn(n_sets * k, 3, dtype=torch.float64, device=device(), generator=g) for _ in range(2))
    a.requires_grad_()
    off = torch.arange(0, n_sets * k + 1, k, device=device())
    best = float("inf")
    for _ in range(6):
        t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        t[0].record()
        superposition_rmsd(a, b, off).sum().backward()
        t[1].record()
        t[1].synchronize()
        best = min(best, t[0].elapsed_time(t[1]))
    return best


@pytest.mark.parametrize("k", [200, 400, 1000])
def test_sets_of_a_wave_go_side_by_side(k):
    """64 sets belong to one wave, a lane each: together they take about as long
    as one, and 64 times as long if they go one after the other."""
    one, all64 = elapsed(1, k), elapsed(64, k)
    print(k, one, all64, flush=True)
    assert all64 < 8.0 * one
