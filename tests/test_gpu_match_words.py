"""The order of the complete matches where their keys are long and level-0 rows
are many: groups of several neighbouring rows, of several templates and
molecules, keys of more than one 64-bit word whose first word is shared, each
by ranking, by the LDS sort and by ranking of listed large groups, against the
oracle's enumeration (patches/Scanner.c.patch:232-334).

Every template atom has a residue name of its own; a molecule has two
interchangeable atoms of each near one point, which give 2^levels matches, and
many more that no partner is in reach of, which make the sets large and the
positions wide."""

import numpy as np
import pytest

from oracle import oracle
from pyjess_amd import Molecule, Template, TemplateAtom, _native

pytestmark = pytest.mark.gpu

RESIDUES = ["GLY", "ALA", "SER", "THR", "VAL", "LEU", "ILE", "PRO", "PHE", "TYR", "TRP", "ASP", "GLU", "HIS"]


def molecule(rng, types, alone):
    """Two near atoms of each type, one of them the first of the molecule and one
    the last, and `alone` far from any other."""
    n = types * (alone + 2)
    kind = np.concatenate([np.arange(types), rng.permutation(np.repeat(np.arange(types), alone)), np.arange(types)])
    side = int(np.ceil(n ** (1 / 3))) + 1
    cell = rng.permutation(side ** 3)[:n]
    xyz = 40.0 * np.stack([cell // side ** 2, cell // side % side, cell % side], axis=1) + 100.0
    near = np.r_[:types, n - types:n]
    spot = rng.permutation(27)[:len(near)]   # about 1 A apart (none nearer than 0.5 A)
    xyz[near] = np.stack([spot // 9, spot // 3 % 3, spot % 3], axis=1) + rng.uniform(-0.2, 0.2, size=(len(near), 3))
    res = np.array([np.frombuffer(r.encode() + b"\0", dtype=np.uint8) for r in RESIDUES])[kind]
    names = np.tile(np.frombuffer(b"_CA_", dtype=np.uint8), (n, 1))
    chains = np.tile(np.frombuffer(b" A", dtype=np.uint8), (n, 1))
    return Molecule.from_arrays(np.round(xyz, 3), names, res, chains, np.arange(1, n + 1), id="WORD")


def template(rng, levels, tid):
    at = [TemplateAtom(chain_id="A", residue_number=i + 1, x=float(x[0]), y=float(x[1]), z=float(x[2]),
                       residue_names=[RESIDUES[i]], atom_names=["CA"], match_mode=0)
          for i, x in enumerate(np.round(rng.uniform(-1.0, 1.0, size=(levels, 3)), 3))]
    return Template(at, id=tid)


# molecules, templates, levels of each, atoms alone per type; then bits that the
# row numbers are shortened by, key words, and whether all groups are ranked,
# sorted in LDS, or (more than 2,048 matches to a row) listed and ranked
CASES = [
    (1, 10, 10, 1500, 0, 2, "ranked"),
    (2, 6, 10, 6001, 1, 3, "ranked"),
    (3, 7, 9, 9000, 2, 2, "ranked"),
    (1, 20, 11, 1500, 0, 2, "sorted"),
    (2, 10, 11, 6001, 1, 3, "sorted"),
    (1, 6, 12, 9000, 0, 3, "sorted"),
    (1, 2, 13, 1100, 0, 3, "listed"),
]


def route(mols, tpls, levels, alone):
    """What the library takes by its sizes."""
    rows = mols * tpls * (alone + 2)
    n = mols * tpls * 2 ** levels
    shift = 0
    while rows >> shift > max(2 * n, 1 << 16):
        shift += 1
    bits = (alone + 2).bit_length()
    first, per = (64 - shift) // bits, 64 // bits
    words = 1 + max(0, -(-(levels - 1 - first) // per))
    group = 2 ** (levels - 1) * (2 if shift else 1)   # a row, with the next template's first
    work = n // group * group * (group - 1) // 2
    way = "ranked" if work <= 8_000_000 and n <= 131072 else "sorted" if group <= 2048 else "listed"
    return n, shift, words, way


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:4])))
@pytest.mark.parametrize("reorder", [True, False])
def test_order(case, reorder):
    n_mols, n_tpls, levels, alone = case[:4]
    got = route(*case[:4])
    print(case, reorder, got, flush=True)
    assert got[1:] == case[4:] and got[0] > 8192
    rng = np.random.default_rng(sum(case[:4]))
    mols = [molecule(rng, levels, alone) for _ in range(n_mols)]
    tpls = [template(rng, levels, f"T{i}") for i in range(n_tpls)]
    ctx = _native.context()
    res = _native.query(_native.TemplateSet(ctx, tpls), _native.MoleculeSet(ctx, mols), 9.0, 8.0, 8.0, 0, reorder)
    pair, rmsd, at = np.asarray(res.pair), np.asarray(res.rmsd), np.asarray(res.atoms)
    assert np.asarray(res.pair_matches).tolist() == [2 ** levels] * (n_mols * n_tpls)
    for m, mol in enumerate(mols):
        stream = oracle.query_stream(mol, tpls, 8.0, 8.0, None, reorder, None)
        want_pair = np.array([w.template for w in stream]) + m * n_tpls
        mine = slice(m * n_tpls * 2 ** levels, (m + 1) * n_tpls * 2 ** levels)
        assert np.array_equal(pair[mine], want_pair)
        assert np.array_equal(rmsd[mine], np.array([w.rmsd for w in stream]))
        assert np.array_equal(at[mine][:, :levels], np.array([w.atoms for w in stream]))
