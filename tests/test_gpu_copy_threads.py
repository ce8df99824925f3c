"""Copies of events and of atom fields from several threads at once, through
the context's shared pinned slots: sizes of one slot, of a few and of more than
all threads' slots hold."""

import threading

import numpy as np
import pytest

from pyjess_amd import _native, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("residues", [40, 9000, 40000])
def test_atom_fields_from_threads(residues):
    print(residues, flush=True)
    rng = np.random.Generator(np.random.PCG64(residues))
    base = synthetic.protein(rng, min(residues, 4000))
    reps = max(1, residues // 4000)
    text = base.dumps().replace("END\n", "").encode() * reps
    ctx = _native.context()
    batch = _native.ParsedMolecules(ctx, [text])
    n = int(batch.atom_offsets()[-1])
    assert n == reps * len(base)
    out = [None] * 4

    def copy(k):
        xyz, serial = np.empty((n, 3)), np.empty(n, dtype=np.int32)
        f = _native.AtomFields(xyz=xyz.ctypes.data, serial=serial.ctypes.data)
        _native._check(_native.lib().jam_molecules_copy_atoms(batch.handle, f))
        out[k] = (xyz, serial)

    threads = [threading.Thread(target=copy, args=(k,)) for k in range(len(out))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for xyz, serial in out:
        assert np.array_equal(xyz, np.tile(base.xyz, (reps, 1)))
        assert np.array_equal(serial, np.tile(base.serial, reps))
