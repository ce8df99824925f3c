"""Where the device parse finds HEADER records (jam_molecules_pdb_headers) and
in which order it indexes atoms, against the host parser: headers before,
between and after models, too many to keep, in texts with bytes above 0x7F and
with each line end; serial numbers that wrap, more residue names than the
small index kernel holds."""

import io

import numpy as np
import pytest

from pyjess_amd import Molecule, _native

pytestmark = pytest.mark.gpu

ATOM = "ATOM  %5d  CA  %-3s A%4d    %8.3f%8.3f%8.3f  1.00  0.00           C"


def atoms(n, serials=None, names=("ALA", "GLY", "ser")):
    serials = range(1, n + 1) if serials is None else serials
    return [ATOM % (s, names[i % len(names)], i % 9999 + 1, i * 0.5, 1.0, -2.0) for i, s in enumerate(serials)]


def header(k):
    return "HEADER    NAME %-35d%02d-JAN-99   %04d" % (k, k % 28 + 1, k % 10000)


TEXTS = {
    "none": atoms(5),
    "first": [header(1)] + atoms(5),
    "late": atoms(3) + [header(7), header(2)] + atoms(2),
    "after the model": atoms(3) + ["ENDMDL", header(3)] + atoms(4),
    "only after": ["HEADER"] + atoms(2) + ["ENDMDL", header(4)],
    "inside a line": ["REMARK HEADER", " HEADER"] + atoms(2),
    "many": [header(k) for k in range(300)] + atoms(2),
    "above 0x7F": ["REMARK éè"] + [header(5)] + atoms(2),
    "empty": [],
}


@pytest.mark.parametrize("end", ["\n", "\r\n", "\r"])
@pytest.mark.parametrize("ignore_endmdl", [False, True])
def test_headers(end, ignore_endmdl):
    datas = [end.join(lines).encode() for lines in TEXTS.values()]
    want = [Molecule.load(io.StringIO(d.decode(), newline=None), device=False, ignore_endmdl=ignore_endmdl) for d in datas]
    singles = [Molecule.load_many([io.BytesIO(d)], ignore_endmdl=ignore_endmdl)[0] for d in datas]
    kept = [k for k, name in enumerate(TEXTS) if name not in ("many", "above 0x7F")]
    batches = [list(range(len(datas))), kept]
    for batch in batches:
        got = Molecule.load_many([io.BytesIO(datas[k]) for k in batch], ignore_endmdl=ignore_endmdl)
        for k, m in zip(batch, got):
            assert (m.id, m.date, m.name, len(m)) == (want[k].id, want[k].date, want[k].name, len(want[k]))
    for m, w in zip(singles, want):
        assert (m.id, m.date, m.name, len(m)) == (w.id, w.date, w.name, len(w))


@pytest.mark.parametrize("serials", ["ascending", "wrapped", "random"])
@pytest.mark.parametrize("names", [3, 257])
def test_index(serials, names):
    rng = np.random.default_rng(names)
    texts = []
    for n in (1, 700, 64, 2500):
        sr = {"ascending": np.arange(n), "wrapped": (np.arange(n) + n // 2) % n, "random": rng.integers(0, 50, size=n)}
        texts.append("\n".join(atoms(n, sr[serials], ["%03X" % k for k in range(names)])).encode())
    host = [Molecule.load(io.StringIO(t.decode()), device=False) for t in texts]
    ctx = _native.context()
    got = _native.ParsedMolecules(ctx, texts).residue_index()
    want = _native.MoleculeSet(ctx, host).residue_index()
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


def test_errors_keep_their_order():
    """A header's own error comes before an atom's."""
    bad_date = "HEADER" + " " * 44 + "99-XXX-99"
    bad_atom = atoms(1)[0][:30] + "  x.x   " + atoms(1)[0][38:]
    with pytest.raises(ValueError, match="time data"):
        Molecule.load_many([io.BytesIO("\n".join([bad_date, bad_atom]).encode())])
    with pytest.raises(ValueError, match="failed to parse atom"):
        Molecule.load_many([io.BytesIO(bad_atom.encode())])
    with pytest.raises(UnicodeDecodeError):
        Molecule.load_many([io.BytesIO(b"REMARK \xff\n" + bad_atom.encode())])
