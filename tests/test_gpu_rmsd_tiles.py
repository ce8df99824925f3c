"""The RMSD kernels' tiles at their edges: sets of 11 to 14 points (up to 12 are
held in registers) mixed in one tile, tiles of exactly 768 points and one more
(the most that LDS holds), 63 to 65 sets, sets of equal size without offsets;
forward and backward, one-sided gradients, against the 50-digit RMSD and
autograd through an SVD on the CPU (the bounds of test_gpu_autograd.py)."""

import numpy as np
import pytest

from oracle.kabsch_torch import kabsch_rmsd_grad
from tests.test_gpu_autograd import device, pairs, run
from tests.test_rmsd_grad_cpu import exact_rmsd

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def check(a, b, off, step):
    w = np.random.default_rng(3).uniform(-1.0, 1.0, size=len(off) - 1)
    r, ga, gb = run(a, b, off, weights=w)
    for s in range(0, len(off) - 1, step):
        A, B = a[off[s]:off[s + 1]], b[off[s]:off[s + 1]]
        want = exact_rmsd(A, B)
        assert abs(r[s] - want) <= 1e-13 * max(1.0, want), s
        _, ta, tb = kabsch_rmsd_grad(A, B)
        x = np.concatenate([ga[off[s]:off[s + 1]], gb[off[s]:off[s + 1]]]).ravel()
        y = w[s] * np.concatenate([ta, tb]).ravel()
        assert np.linalg.norm(x - y) <= 1e-10 * np.linalg.norm(y), s


@pytest.mark.parametrize("sizes", [[3], [11], [12], [13], [12, 13], [3, 14, 12, 30, 4], [6, 24]])
@pytest.mark.parametrize("n_sets", [1, 63, 64, 65, 130])
def test_sizes(sizes, n_sets):
    print(sizes, n_sets, flush=True)
    a, b, _ = pairs(n_sets, 5, k_min=max(sizes), k_max=max(sizes), collinear=0.0)
    k = np.array([sizes[s % len(sizes)] for s in range(n_sets)])
    keep = np.concatenate([np.arange(x) + s * max(sizes) for s, x in enumerate(k)])
    check(np.ascontiguousarray(a[keep]), np.ascontiguousarray(b[keep]),
          np.concatenate([[0], np.cumsum(k)]).astype(np.int64), 1 + n_sets // 20)


@pytest.mark.parametrize("extra", [0, 1])
def test_full_tile(extra):
    a, b, off = pairs(64, 6, k_min=13, k_max=13, collinear=0.0)
    k = np.full(64, 12)
    k[10] += extra
    keep = np.concatenate([np.arange(x) + 13 * s for s, x in enumerate(k)])
    check(np.ascontiguousarray(a[keep]), np.ascontiguousarray(b[keep]),
          np.concatenate([[0], np.cumsum(k)]).astype(np.int64), 3)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("k", [3, 12, 13])
def test_equal_sizes_one_side(side, k):
    from pyjess_amd.autograd import superposition_rmsd

    a, b, off = pairs(70, 7, k_min=k, k_max=k, collinear=0.0)
    r2, *both = run(a, b, off)
    t = [torch.tensor(x.reshape(70, k, 3), device=device(), requires_grad=q == side) for q, x in enumerate((a, b))]
    r = superposition_rmsd(*t)
    r.sum().backward()
    assert np.array_equal(r.detach().cpu().numpy(), r2)
    assert np.array_equal(t[side].grad.cpu().numpy().reshape(-1, 3), both[side])
    with torch.no_grad():
        z = torch.zeros(5, 0, 3, dtype=torch.float64, device=device())
        assert superposition_rmsd(z, z).tolist() == [0.0] * 5
