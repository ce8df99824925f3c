"""The residue-name index of molecules uploaded from host arrays
(jam_molecules_create) against a stable sort by (upper-cased name, serial),
patches/ResIndex.c.patch:18-26,34-119: atom counts around the 64 lanes of a
wave and the 1,024 threads of a workgroup, names in mixed case, one name, more
names than the device kernel holds, serial numbers that ascend, wrap, descend
or repeat, alone and in one batch."""

import numpy as np
import pytest

from pyjess_amd import _native

pytestmark = pytest.mark.gpu


class Arrays:
    """What MoleculeSet reads of a molecule."""

    def __init__(self, rng, n, n_names, serial):
        letters = np.frombuffer(b"AbCdEfGhIjKlMnOp", dtype=np.uint8)
        names = np.zeros((max(n_names, 1), 4), dtype=np.uint8)
        for d in range(3):
            names[:, d] = letters[(np.arange(len(names)) >> (4 * d)) % 16]
        run = np.repeat(rng.integers(0, len(names), size=n // 7 + 1), 7)[:n]
        self.resnames = names[run]
        flip = rng.random(n) < 0.3
        lower = (self.resnames >= 65) & (self.resnames <= 90) & flip[:, None]
        self.resnames = np.where(lower, self.resnames + 32, self.resnames).astype(np.uint8)
        self.xyz = rng.normal(size=(n, 3))
        self.names = np.full((n, 4), 65, dtype=np.uint8)
        self.chains = np.full((n, 2), 65, dtype=np.uint8)
        self.resseq = np.arange(n, dtype=np.int32)
        self.serial = {
            "ascending": np.arange(n), "equal": np.zeros(n), "wrapped": (np.arange(n) + n // 3) % max(n, 1),
            "descending": -np.arange(n), "random": rng.integers(-5, 5, size=n),
        }[serial].astype(np.int32)

    def __len__(self):
        return len(self.xyz)

    def index(self):
        up = self.resnames.astype(np.uint32)
        up = np.where((up >= 97) & (up <= 122), up - 32, up)
        key = up[:, 0] | (up[:, 1] << 8) | (up[:, 2] << 16) | (up[:, 3] << 24)
        perm = np.lexsort((np.arange(len(key)), self.serial, key))
        keys, begin = np.unique(key[perm], return_index=True)
        return perm, keys, begin, np.append(begin[1:], len(key))[:len(keys)]


def check(mols):
    perm, off, key, begin, end = _native.MoleculeSet(_native.context(), mols).residue_index()
    want = [m.index() for m in mols]
    assert off.tolist() == np.cumsum([0] + [len(w[1]) for w in want]).tolist()
    for got, k in ((perm, 0), (key, 1), (begin, 2), (end, 3)):
        assert np.array_equal(got, np.concatenate([w[k] for w in want]))


@pytest.mark.parametrize("serial", ["ascending", "equal", "wrapped", "descending", "random"])
@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 1023, 1024, 1025, 20011])
def test_one_molecule(n, serial):
    print(n, serial, flush=True)
    check([Arrays(np.random.default_rng(n), n, 21, serial)])


@pytest.mark.parametrize("n_names", [1, 2, 255, 256, 257, 2500])
def test_number_of_names(n_names):
    print(n_names, flush=True)
    check([Arrays(np.random.default_rng(n_names), 30000, n_names, "ascending")])


@pytest.mark.parametrize("serials", [("ascending",), ("ascending", "random", "wrapped")])
def test_batch(serials):
    rng = np.random.default_rng(5)
    sizes = [0, 3000, 64, 1, 0, 4097, 1025, 700] * 6
    check([Arrays(rng, n, 300 if len(serials) > 1 and i == 13 else 25, serials[i % len(serials)])
           for i, n in enumerate(sizes)])


def test_large_upload():
    """More than the two pinned halves hold."""
    rng = np.random.default_rng(6)
    mols = [Arrays(rng, n, 25, "ascending") for n in (400003, 350001, 5, 300011)]
    check(mols)
    mset = _native.MoleculeSet(_native.context(), mols)
    n = int(mset.atom_offsets()[-1])
    fields = {"xyz": np.empty((n, 3)), "names": np.empty((n, 4), dtype=np.uint8),
              "resnames": np.empty((n, 4), dtype=np.uint8), "resseq": np.empty(n, dtype=np.int32)}
    f = _native.AtomFields(**{k: v.ctypes.data for k, v in fields.items()})
    _native._check(_native.lib().jam_molecules_copy_atoms(mset.handle, f))
    for k, v in fields.items():
        assert np.array_equal(v, np.concatenate([getattr(m, k) for m in mols])), k
