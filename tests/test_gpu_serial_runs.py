"""The residue-name index of molecules whose serial numbers descend at a few
atoms, as they do where the five columns of a PDB text wrap: uploaded and
parsed, against a stable sort by (upper-cased name, serial)
(patches/ResIndex.c.patch:18-26,34-119). Up to 64 such atoms in a batch go
one way, more another."""

import time

import numpy as np
import pytest

from pyjess_amd import Molecule, _native
from tests.test_gpu_residue_index import Arrays, check

pytestmark = pytest.mark.gpu


def serials(rng, n, down):
    """n serial numbers with repeats that descend at `down` atoms."""
    s = np.cumsum(rng.integers(0, 3, size=n))
    for i in np.sort(rng.choice(np.arange(1, n), size=down, replace=False)):
        s[i:] -= s[i] - s[i - 1] + rng.integers(1, 9)
    return s.astype(np.int32)


def molecule(seed, n, down):
    m = Arrays(np.random.default_rng(seed), n, 21, "ascending")
    m.serial = serials(np.random.default_rng(seed + 1), n, down)
    assert np.count_nonzero(np.diff(m.serial) < 0) == down
    return m


@pytest.mark.parametrize("down", [1, 2, 21, 63, 64, 65])
@pytest.mark.parametrize("n", [66, 1024, 20011])
def test_one_molecule(n, down):
    print(n, down, flush=True)
    check([molecule(n, n, down)])


def test_batch():
    sizes = [(3, 1), (3000, 9), (2, 1), (64, 0), (0, 0), (4097, 30), (700, 1)]
    check([molecule(k, n, d) if n > 1 else Arrays(np.random.default_rng(k), n, 21, "ascending")
           for k, (n, d) in enumerate(sizes)])
    check([molecule(k, n, d) if n > 1 else Arrays(np.random.default_rng(k), n, 21, "ascending")
           for k, (n, d) in enumerate(sizes * 2)])


def text(mol):
    xyz = np.round(np.abs(mol.xyz) + 1.0, 3)
    names = np.tile(np.frombuffer(b"_CA_", dtype=np.uint8), (len(mol), 1))
    names[:, 3] = ord("_")
    return Molecule.from_arrays(xyz, names, mol.resnames, mol.chains, mol.resseq % 9000,
                                mol.serial - mol.serial.min() + 1).dumps().encode()


@pytest.mark.parametrize("downs", [(1,), (64,), (65,), (2, 0, 5), (40, 25, 0)])
def test_texts(downs):
    mols = [molecule(31 + k, 3000 + 64 * k, d) for k, d in enumerate(downs)]
    batch = _native.ParsedMolecules(_native.context(), [text(m) for m in mols])
    got = np.empty(sum(map(len, mols)), dtype=np.int32)
    f = _native.AtomFields(serial=got.ctypes.data)
    _native._check(_native.lib().jam_molecules_copy_atoms(batch.handle, f))
    assert np.array_equal(got, np.concatenate([m.serial - m.serial.min() + 1 for m in mols]))
    perm = batch.residue_index()[0]
    assert np.array_equal(perm, np.concatenate([m.index()[0] for m in mols]))


@pytest.mark.parametrize("n,down", [(400000, "wrapped"), (100000, "reversed")])
def test_upload_time(n, down):
    """Serial numbers that descend cost an upload little: nothing is sorted on
    the host."""
    times = []
    for serial in (np.arange(n), np.arange(n) % 99999 if down == "wrapped" else np.arange(n, 0, -1)):
        m = Arrays(np.random.default_rng(1), n, 21, "ascending")
        m.serial = serial.astype(np.int32)
        best = float("inf")
        for _ in range(5):
            t0 = time.perf_counter()
            _native.MoleculeSet(_native.context(), [m])
            best = min(best, time.perf_counter() - t0)
        times.append(best)
    print(times, flush=True)
    assert times[1] < 2.5 * times[0]
