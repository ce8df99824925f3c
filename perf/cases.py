"""Representative calls of this package, for timing it and comparing its results.

Search: the drop-in ``Jess.query`` (one molecule, hits read as they come),
``Jess.query_batch`` over freshly built molecules, and the C ABI
(``include/jess_amd.h`` through its ctypes binding) over molecules and
templates resident in HBM, the events copied to host arrays. Beside it: the
differentiable superposition RMSD (forward and backward), the batched
superposition of host arrays, and PDB text to molecules.

Proteins and templates come from ``pyjess_amd.synthetic`` (self-avoiding CA
walks, real residue and atom names, coordinates rounded to 0.001 A as in PDB
files, so that equal coordinates occur); the CA walks and a stock of random
templates are the same for every seed, residue types, side chains, planted
templates and the choice among the stock come from the seed.
"""

import ctypes
import functools
import io
import itertools
import math

import numpy as np
import torch

from pyjess_amd import Jess, Molecule, _native, synthetic
from pyjess_amd.autograd import superposition_rmsd

ATOMS_PER_RESIDUE = 8.35   # synthetic.protein, on average


def listed():
    return [
        # one small protein against a handful of three-residue templates: the
        # smallest call a user makes, where launches and latency count
        {"name": "query-2k", "kind": "query", "residues": 250, "chains": 1, "templates": 10, "res_min": 3,
         "res_max": 3, "planted": 0.3, "cutoff": 1.5, "ignore_chain": "", "best_match": False, "reorder": True,
         "cap": 0},
        # the everyday drop-in call: one protein against a template library
        {"name": "query-8k", "kind": "query", "residues": 1000, "chains": 1, "templates": 500, "res_min": 3,
         "res_max": 6, "planted": 0.3, "cutoff": 1.5, "ignore_chain": "", "best_match": False, "reorder": True,
         "cap": 10000},
        # a large multi-chain complex, chains ignored in the residue test, a
        # wider cutoff, one best hit per template, in the template's own order
        {"name": "query-40k", "kind": "query", "residues": 4801, "chains": 8, "templates": 300, "res_min": 2,
         "res_max": 8, "planted": 0.1, "cutoff": 2.0, "ignore_chain": "residues", "best_match": True,
         "reorder": False, "cap": 0},
        # a structure file as it arrives (just above the size that is parsed
        # on the device), loaded and searched: the whole drop-in program
        {"name": "load-query-16k", "kind": "load_query", "atoms": 16003, "chains": 2, "templates": 100,
         "res_min": 3, "res_max": 6, "planted": 0.2, "cutoff": 1.5},
        # many new proteins at once through the batched drop-in
        {"name": "batch-256", "kind": "batch", "molecules": 256, "median": 4000, "templates": 200, "res_min": 3,
         "res_max": 6, "planted": 0.1, "cutoff": 1.5, "cap": 10000},
        # a proteome resident in HBM, screened against a set of templates
        {"name": "screen-768", "kind": "screen", "molecules": 768, "median": 4000, "templates": 200, "res_min": 3,
         "res_max": 6, "planted": 0.1, "symmetric": 0.0, "cutoff": 1.5, "all_fields": True},
        # one large assembly against a thousand templates, every event field
        # copied out
        {"name": "screen-1x100k", "kind": "screen", "molecules": 1, "median": 100000, "templates": 1000,
         "res_min": 2, "res_max": 8, "planted": 0.1, "symmetric": 0.2, "cutoff": 2.5, "all_fields": True},
        # a stretch of a library-scale search: assemblies resident in HBM,
        # millions of events, their pairs, flags and RMSDs copied out
        {"name": "screen-6x100k", "kind": "screen", "molecules": 6, "median": 100000, "templates": 2000,
         "res_min": 2, "res_max": 8, "planted": 0.1, "symmetric": 0.2, "cutoff": 2.5, "all_fields": False},
        # the loss of a small fit: forward and backward, launch-bound
        {"name": "grad-256", "kind": "grad", "sets": 256, "k_min": 8, "k_max": 8},
        # training scale: ragged sets of 3 to 12 points, some nearly collinear
        {"name": "grad-1m", "kind": "grad", "sets": 1000000, "k_min": 3, "k_max": 12},
        # superposition of matched point sets held in host memory
        {"name": "superpose-20k", "kind": "superpose", "sets": 20011, "k": 8},
        # a directory of large structure files read into molecules
        {"name": "load-4x100k", "kind": "load", "texts": 4, "atoms": 100001, "chains": 20},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["query", "query", "query", "batch", "screen", "screen", "assemblies", "grad", "grad",
                       "superpose", "load", "load_query"])
    res_min = rng.randint(2, 3)
    res_max = rng.randint(res_min + 1, 8)
    if kind == "query":
        return {"kind": "query", "residues": _log_uniform(rng, 150, 4801), "chains": rng.randint(1, 8),
                "templates": _log_uniform(rng, 7, 500), "res_min": res_min, "res_max": res_max,
                "planted": round(rng.uniform(0.05, 0.3), 2), "cutoff": rng.choice([1.0, 1.5, 2.0]),
                "ignore_chain": rng.choice(["", "residues", "atoms"]), "best_match": rng.random() < 0.4,
                "reorder": rng.random() < 0.7, "cap": rng.choice([0, 100, 10000])}
    if kind == "load_query":
        return {"kind": "load_query", "atoms": _log_uniform(rng, 14000, 40000), "chains": rng.randint(1, 8),
                "templates": _log_uniform(rng, 7, 300), "res_min": 3, "res_max": 6, "planted": 0.2, "cutoff": 1.5}
    if kind == "batch":
        return {"kind": "batch", "molecules": _log_uniform(rng, 5, 256), "median": _log_uniform(rng, 1000, 4000),
                "templates": _log_uniform(rng, 11, 200), "res_min": res_min, "res_max": min(res_max, 6),
                "planted": 0.1, "cutoff": 1.5, "cap": rng.choice([0, 100, 10000])}
    if kind == "screen":
        return {"kind": "screen", "molecules": _log_uniform(rng, 11, 768), "median": _log_uniform(rng, 1000, 4000),
                "templates": _log_uniform(rng, 11, 200), "res_min": 3, "res_max": 6, "planted": 0.1,
                "symmetric": 0.0, "cutoff": rng.choice([1.5, 2.0]), "all_fields": True}
    if kind == "assemblies":
        return {"kind": "screen", "molecules": rng.randint(1, 4), "median": _log_uniform(rng, 30000, 100000),
                "templates": _log_uniform(rng, 101, 1500), "res_min": 2, "res_max": 8, "planted": 0.1,
                "symmetric": 0.2, "cutoff": rng.choice([1.5, 2.0, 2.5]), "all_fields": rng.random() < 0.3}
    if kind == "grad":
        k_min = rng.randint(3, 8)
        return {"kind": "grad", "sets": _log_uniform(rng, 33, 1000000), "k_min": k_min,
                "k_max": rng.choice([k_min, k_min + rng.randint(1, 12 - k_min)])}
    if kind == "superpose":
        return {"kind": "superpose", "sets": _log_uniform(rng, 101, 20011), "k": rng.randint(4, 24)}
    return {"kind": "load", "texts": rng.randint(1, 4), "atoms": _log_uniform(rng, 16001, 100001),
            "chains": rng.randint(1, 20)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _walk():
    """One long self-avoiding CA walk: any stretch of it is one, too."""
    return synthetic.ca_walk(np.random.Generator(np.random.PCG64(71)), 16000)


@functools.lru_cache(maxsize=None)
def _stock(res_min, res_max, symmetric):
    """Random templates of a library, drawn from by every seed."""
    rng = np.random.Generator(np.random.PCG64(74))
    return synthetic.template_set(rng, [], 600, 0.0, (res_min, res_max), (2, 3), p_symmetric=symmetric)


def _rng(case, seed):
    return np.random.Generator(np.random.PCG64([seed, 73]))


def _protein(rng, residues, chains):
    walk = _walk()
    start = int(rng.integers(0, len(walk) - residues + 1))
    return synthetic.protein(rng, residues, n_chains=chains, mol_id="SYNT", ca=walk[start:start + residues])


def _templates(rng, mols, case):
    """``templates`` of them in random order: planted ones copied from the
    molecules with noise, the others from the stock (in new positions of the
    list, again and again where the stock is smaller)."""
    n = case["templates"]
    n_planted = int(round(case["planted"] * n))
    residues = (case["res_min"], case["res_max"])
    symmetric = case.get("symmetric", 0.0)
    out = synthetic.template_set(rng, mols, n_planted, 1.0, residues, (2, 3), p_symmetric=symmetric)
    stock = _stock(*residues, symmetric)
    while len(out) < n:
        out += [stock[i] for i in rng.permutation(len(stock))[:n - len(out)]]
    return [out[i] for i in rng.permutation(n)]


def _molecules(rng, case):
    """Assemblies of 20 chains, or proteins of lognormal sizes: stretches of a
    long chain, each in an orientation of its own."""
    if case["median"] >= 30000:
        residues = int(round(case["median"] / 8.05))
        return [_protein(rng, residues, 20) for _ in range(case["molecules"])]
    base = _protein(rng, 12000, 1)
    first = np.concatenate([[0], np.flatnonzero(np.diff(base.resseq)) + 1, [len(base)]])
    sizes = np.clip(np.exp(rng.normal(math.log(case["median"]), 0.6, size=case["molecules"])), 500, 40000)
    rotations = synthetic.random_rotations(rng, case["molecules"])
    out = []
    for i, size in enumerate(sizes):
        residues = max(3, int(size / ATOMS_PER_RESIDUE))
        r0 = int(rng.integers(0, 12000 - residues + 1))
        a, b = int(first[r0]), int(first[r0 + residues])
        xyz = np.round(base.xyz[a:b] @ rotations[i].T, 3)
        out.append(Molecule.from_arrays(xyz, base.names[a:b], base.resnames[a:b], base.chains[a:b],
                                        base.resseq[a:b] - base.resseq[a] + 1, id="M%04d" % i,
                                        element=base.element[a:b]))
    return out


def _text(rng, case):
    """A protein of ``atoms`` atoms and its PDB text (moved to positive
    coordinates; five serial columns, so serial numbers wrap)."""
    n = case["atoms"]
    mol = _protein(rng, n // 8 + 40, case["chains"])
    while len(mol) < n:
        mol = _protein(rng, n // 8 + 40, case["chains"])
    xyz = np.round(mol.xyz[:n] - mol.xyz[:n].min(axis=0) + 1.0, 3)
    serial = (np.arange(n) % 99999 + 1).astype(np.int32)
    moved = Molecule.from_arrays(xyz, mol.names[:n], mol.resnames[:n], mol.chains[:n], mol.resseq[:n], serial,
                                 id="SYNT", element=mol.element[:n])
    return moved, moved.dumps().encode()


def _point_sets(case, seed):
    """Pairs of point sets (a, b, offsets) on the GPU: a is a stretch of a
    jagged chain, b its rotated and moved copy with noise of 0.5 A; one ragged
    set in fifty is three nearly collinear points."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    f64 = dict(dtype=torch.float64, device="cuda")
    n, k_min, k_max = case["sets"], case["k_min"], case["k_max"]
    # as many sets of each size, and of lines, for every seed
    line = torch.arange(n, device="cuda") < (n // 50 if k_min < k_max else 0)
    k = torch.where(line, 3, k_min + torch.arange(n, device="cuda") % (k_max - k_min + 1))
    order = torch.randperm(n, generator=g, device="cuda")
    line, k = line[order], k[order]
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(k, 0)
    total = int(off[-1])
    owner = torch.repeat_interleave(torch.arange(n, device="cuda"), k, output_size=total)
    local = (torch.arange(total, device="cuda") - off[owner]).to(torch.float64)[:, None]
    axis = torch.nn.functional.normalize(torch.randn(n, 3, generator=g, **f64), dim=1)
    scatter = torch.where(line, 0.02, 1.2)[:, None].to(torch.float64)
    origin = 30.0 * torch.randn(n, 3, generator=g, **f64)
    a = origin[owner] + 1.5 * local * axis[owner] + scatter[owner] * torch.randn(total, 3, generator=g, **f64)
    q = torch.nn.functional.normalize(torch.randn(n, 4, generator=g, **f64), dim=1)
    u, w = q[owner, 1:], q[owner, :1]
    turned = a + 2.0 * torch.linalg.cross(u, torch.linalg.cross(u, a) + w * a)
    shift = 10.0 * torch.randn(n, 3, generator=g, **f64)
    b = turned + shift[owner] + 0.5 * torch.randn(total, 3, generator=g, **f64)
    weight = torch.rand(n, generator=g, **f64)
    return a.contiguous(), b.contiguous(), off, weight


def _rows(case):
    """Rows of the program's result buffers: more than a search of this size
    finds (a buffer too small is grown)."""
    if case["kind"] == "screen":
        dense = 0.012 * case["median"] if case["median"] >= 30000 else 1.0
        return int(case["molecules"] * case["templates"] * dense) + 4096
    if case["kind"] == "batch":
        return 8 * case["molecules"] * case["templates"] + 4096
    atoms = case.get("atoms") or case["residues"] * ATOMS_PER_RESIDUE
    return int(case["templates"] * (32 + 0.01 * atoms))


def prepare(case, seed):
    kind = case["kind"]
    rng = _rng(case, seed)
    state = {"case": case}
    if kind in ("query", "load_query", "batch"):
        state["rmsd"] = np.zeros(_rows(case), dtype=np.float64)
    if kind == "query":
        mol = _protein(rng, case["residues"], case["chains"])
        state["molecule"] = mol
        state["jess"] = Jess(_templates(rng, [mol], case))
    elif kind == "load_query":
        mol, state["text"] = _text(rng, case)
        n = int(np.flatnonzero(np.diff(mol.resseq))[-1]) + 1   # templates come from whole residues
        whole = Molecule.from_arrays(mol.xyz[:n], mol.names[:n], mol.resnames[:n], mol.chains[:n], mol.resseq[:n])
        state["jess"] = Jess(_templates(rng, [whole], case))
    elif kind == "batch":
        mols = _molecules(rng, case)
        state["molecules"] = mols
        state["jess"] = Jess(_templates(rng, mols, case))
    elif kind == "screen":
        mols = _molecules(rng, case)
        ctx = _native.context()
        state["ctx"] = ctx
        state["templates"] = _native.TemplateSet(ctx, _templates(rng, mols, case))
        state["molecules"] = _native.MoleculeSet(ctx, mols)
        state["params"] = _native.Params(2.0, case["cutoff"], case["cutoff"], 0, 1)
        state["events"] = {}
    elif kind == "grad":
        a, b, off, weight = _point_sets(case, seed)
        if case["k_min"] == case["k_max"]:
            a, b, off = a.view(case["sets"], -1, 3), b.view(case["sets"], -1, 3), None
        state.update(a=a.requires_grad_(), b=b.requires_grad_(), off=off, weight=weight)
    elif kind == "superpose":
        a, b, _, _ = _point_sets({"sets": case["sets"], "k_min": case["k"], "k_max": case["k"]}, seed)
        state["a"] = a.view(case["sets"], -1, 3).cpu().numpy()
        state["b"] = b.view(case["sets"], -1, 3).cpu().numpy()
    elif kind == "load":
        state["texts"] = [_text(rng, case)[1] for _ in range(case["texts"])]
    else:
        raise ValueError(kind)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _read(state, hits):
    """Reads the RMSD of every hit into the program's buffer, whose unused end
    stays zero."""
    found = [h.rmsd for h in hits]
    if len(found) > len(state["rmsd"]):
        state["rmsd"] = np.zeros(len(found), dtype=np.float64)
    state["rmsd"][:len(found)] = found
    return state["rmsd"]


# event fields of jam_result_copy: values per event and their type
_FIELDS = {"pair": (1, np.int32), "rank": (1, np.int64), "flag": (1, np.int32), "rmsd": (1, np.float64),
           "rotation": (9, np.float64), "c0": (3, np.float64), "c1": (3, np.float64), "atoms": (0, np.int32)}


def _screen(state):
    """jam_query over resident molecules and templates, the events copied into
    host arrays that the program keeps and grows."""
    L = _native.lib()
    ctx, keep = state["ctx"], state["events"]
    wanted = list(_FIELDS) if state["case"]["all_fields"] else ["pair", "flag", "rmsd"]
    h = ctypes.c_void_p()
    with ctx.lock:
        _native._check(L.jam_query(ctx.handle, state["templates"].handle, state["molecules"].handle,
                                   ctypes.byref(state["params"]), ctypes.byref(h)))
        try:
            n, stride = L.jam_result_n_events(h), L.jam_result_stride(h)
            if not keep or keep["pair"].shape[0] < n:
                for name in wanted:
                    width, dtype = _FIELDS[name]
                    # room for the widest rows (up to three atoms a residue)
                    width = width or max(stride, 3 * state["case"]["res_max"])
                    keep[name] = np.zeros((max(n, _rows(state["case"])), width), dtype=dtype)
                keep["matches"] = np.zeros(L.jam_result_n_pairs(h), dtype=np.int64)
            _native._check(L.jam_result_copy(h, *(keep[f].ctypes.data if f in keep else None for f in _FIELDS)))
            _native._check(L.jam_result_pair_matches(h, keep["matches"].ctypes.data))
        finally:
            L.jam_result_free(h)
    return keep


def _atom_arrays(mols):
    fields = ("xyz", "names", "resnames", "chains", "resseq", "serial", "altloc", "icode", "occupancy", "tempfactor",
              "segid", "element", "charge")
    return [{f: getattr(m, f) for f in fields} for m in mols]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "query":
        hits = list(state["jess"].query(
            state["molecule"], 2.0, case["cutoff"], case["cutoff"], max_candidates=case["cap"] or None,
            ignore_chain=case["ignore_chain"] or None, best_match=case["best_match"], reorder=case["reorder"]))
        return _read(state, hits)
    if kind == "load_query":
        mol = Molecule.load(io.BytesIO(state["text"]))
        hits = list(state["jess"].query(mol, 2.0, case["cutoff"], case["cutoff"]))
        return {"rmsd": _read(state, hits), "xyz": mol.xyz}
    if kind == "batch":
        found = state["jess"].query_batch(state["molecules"], 2.0, case["cutoff"], case["cutoff"],
                                          max_candidates=case["cap"] or None)
        return {"hits": np.array([len(h) for h in found]), "rmsd": _read(state, itertools.chain(*found))}
    if kind == "screen":
        return _screen(state)
    if kind == "grad":
        a, b = state["a"], state["b"]
        rmsd = superposition_rmsd(a, b, state["off"])
        grad_a, grad_b = torch.autograd.grad(rmsd, (a, b), state["weight"])
        return {"rmsd": rmsd.detach(), "grad_a": grad_a, "grad_b": grad_b}
    if kind == "superpose":
        rmsd, rotation, c0, c1 = _native.superpose_batch(state["a"], state["b"])
        return {"rmsd": rmsd, "rotation": rotation, "c0": c0, "c1": c1}
    return _atom_arrays(Molecule.load_many([io.BytesIO(t) for t in state["texts"]]))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Search: every atom (coordinates, names, chain, residue number: 40 bytes)
    and every template (32 bytes an atom and its distances) read once, the
    match count of every pair written, and of every atom and template the
    three plane tests of about 8 flops that one annulus takes. Superposition:
    the points read, the results written, 27 flops a point and about 1100 an
    eigenproblem. Text: 80 bytes an atom read, 66 written."""
    kind = case["kind"]
    if kind in ("query", "load_query", "batch", "screen"):
        if kind in ("query", "load_query"):
            mols, atoms = 1, case.get("atoms") or case["residues"] * ATOMS_PER_RESIDUE
        else:
            mols = case["molecules"]
            atoms = mols * case["median"] * (1.2 if case["median"] < 30000 else 1.04)
        n = 1.25 * (case["res_min"] + case["res_max"])
        pairs = mols * case["templates"]
        text = 146.0 * atoms if kind == "load_query" else 0.0
        return {"bytes": 40.0 * atoms + case["templates"] * (32 * n + 8 * n * n) + 8.0 * pairs + text,
                "flops": 8.0 * n * atoms / 160.0 * case["templates"]}
    if kind == "grad":
        points = case["sets"] * 0.5 * (case["k_min"] + case["k_max"])
        return {"bytes": 96.0 * points + 24.0 * case["sets"], "flops": 110.0 * points + 1100.0 * case["sets"]}
    if kind == "superpose":
        points = float(case["sets"] * case["k"])
        return {"bytes": 48.0 * points + 128.0 * case["sets"], "flops": 27.0 * points + 1100.0 * case["sets"]}
    atoms = case["texts"] * case["atoms"]
    return {"bytes": 146.0 * atoms, "flops": 0.0}


# ---------------------------------------------------------------------------
# the same in 64 bits, without the package's kernels
# ---------------------------------------------------------------------------

def _kabsch(a, b, off):
    """RMSD, rotation, residuals' parts of every set, by numpy's SVD."""
    k = np.diff(off)
    owner = np.repeat(np.arange(len(k)), k)
    ca = np.add.reduceat(a, off[:-1]) / k[:, None]
    cb = np.add.reduceat(b, off[:-1]) / k[:, None]
    A, B = a - ca[owner], b - cb[owner]
    X = np.add.reduceat(B[:, :, None] * A[:, None, :], off[:-1])
    U, _, Vt = np.linalg.svd(X)
    D = np.ones((len(k), 3))
    D[:, 2] = np.sign(np.linalg.det(U) * np.linalg.det(Vt))
    R = (U * D[:, None, :]) @ Vt
    RA = (R[owner] @ A[:, :, None])[:, :, 0]
    RtB = (R[owner].transpose(0, 2, 1) @ B[:, :, None])[:, :, 0]
    rmsd = np.sqrt(np.add.reduceat(((B - RA) ** 2).sum(axis=1), off[:-1]) / k)
    return rmsd, R, ca, cb, A - RtB, B - RA, owner, k


def exact(case, seed):
    kind = case["kind"]
    if kind == "grad":
        a, b, off, weight = (t.cpu().numpy() for t in _point_sets(case, seed))
        rmsd, _, _, _, ra, rb, owner, k = _kabsch(a, b, off)
        scale = (weight / (k * rmsd))[owner][:, None]
        ga, gb = ra * scale, rb * scale
        if case["k_min"] == case["k_max"]:
            ga, gb = ga.reshape(case["sets"], -1, 3), gb.reshape(case["sets"], -1, 3)
        return {"rmsd": rmsd, "grad_a": ga, "grad_b": gb}
    if kind == "superpose":
        a, b, off, _ = (t.cpu().numpy() for t in
                        _point_sets({"sets": case["sets"], "k_min": case["k"], "k_max": case["k"]}, seed))
        rmsd, R, ca, cb = _kabsch(a, b, off)[:4]
        return {"rmsd": rmsd, "rotation": R, "c0": ca, "c1": cb}
    if kind == "load":
        rng = _rng(case, seed)
        none = dict.fromkeys(("names", "resnames", "chains", "resseq", "serial", "altloc", "icode", "segid",
                              "element", "charge"))
        mols = [_text(rng, case)[0] for _ in range(case["texts"])]
        return [{"xyz": m.xyz, "occupancy": np.ones(len(m), dtype=np.float64),
                 "tempfactor": np.zeros(len(m), dtype=np.float64), **none} for m in mols]
    if kind == "load_query":
        return {"rmsd": None, "xyz": _text(_rng(case, seed), case)[0].xyz}
    # the RMSDs of a search come in the visit order of the reference's
    # kd-trees, which no plain library call gives
    return None
