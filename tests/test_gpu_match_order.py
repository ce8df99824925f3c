"""The order of the complete matches of a query: by groups of level-0 rows, or
by radix passes where a row has too many matches, against the oracle's
enumeration (patches/Scanner.c.patch:232-334). Clusters of interchangeable
atoms, in which every ordered choice of atoms is a match: below and above
the sizes that each way of sorting takes; templates of one to five atoms, several molecules, so that matches of
several templates share a group."""

import numpy as np
import pytest

from oracle import oracle
from pyjess_amd import Jess, Molecule, Template, TemplateAtom, _native

pytestmark = pytest.mark.gpu


def cluster(rng, n, radius):
    xyz = np.round(rng.uniform(-radius, radius, size=(n, 3)), 3)
    names = np.tile(np.frombuffer(b"_CA_", dtype=np.uint8), (n, 1))
    res = np.tile(np.frombuffer(b"GLY\0", dtype=np.uint8), (n, 1))
    chains = np.tile(np.frombuffer(b" A", dtype=np.uint8), (n, 1))
    return Molecule.from_arrays(xyz, names, res, chains, np.arange(1, n + 1), id="CLUS")


def template(k, tid):
    at = [TemplateAtom(chain_id="A", residue_number=i + 1, x=1.5 * i, y=0.4 * (i % 2), z=0.0,
                       residue_names=["GLY"], atom_names=["CA"], match_mode=0) for i in range(k)]
    return Template(at, id=tid)


@pytest.mark.parametrize("atoms,sizes", [
    ((12,), (4,)),                  # under 11,880 matches, 990 to a row: ranking
    ((23, 24, 25), (1, 2, 3)),      # groups of several templates and molecules
    ((9, 10), (5, 1, 4)),           # two key words' worth of levels, one-atom templates
    ((15, 17, 14), (4, 3)),         # 2,184 and 3,360 to a row: more than the LDS sort takes
    ((14,) * 12 + (15,), (4,)),     # the same beside smaller groups, LDS sort and ranking
    ((14,) * 40, (4, 3, 4)),        # 1.3 M, at most 1,716 to a row: LDS sort
    ((44,), (4,)),                  # 79,464 to a row: radix passes
])
@pytest.mark.parametrize("reorder", [True, False])
def test_order(atoms, sizes, reorder):
    print(atoms, sizes, reorder, flush=True)
    rng = np.random.default_rng(sum(atoms))
    mols = [cluster(rng, n, 1.2) for n in atoms]
    tpls = [template(k, f"T{i}") for i, k in enumerate(sizes)]
    ctx = _native.context()
    res = _native.query(_native.TemplateSet(ctx, tpls), _native.MoleculeSet(ctx, mols), 1.1, 8.0, 8.0, 0, reorder)
    pair, rmsd, at = np.asarray(res.pair), np.asarray(res.rmsd), np.asarray(res.atoms)
    e = 0
    for m, mol in enumerate(mols):
        stream = oracle.query_stream(mol, tpls, 8.0, 8.0, None, reorder, None)
        want = [(w.template, w.rmsd, tuple(w.atoms)) for w in stream if w.rmsd <= 1.1]
        n = int(np.count_nonzero(pair // len(tpls) == m))
        got = [(int(pair[k] % len(tpls)), float(rmsd[k]), tuple(x for x in at[k].tolist() if x >= 0))
               for k in range(e, e + n)]
        assert len(want) > 100
        assert got == want
        counts = np.bincount([w.template for w in stream], minlength=len(tpls))
        assert np.asarray(res.pair_matches).reshape(len(mols), -1)[m].tolist() == counts.tolist()
        e += n
