"""The kd kernels as the library launches them (kd_launches in
pyjess_amd/csrc/jam_kd.h), run on the CPU under the emulation of tests/emu/ with
AddressSanitizer and UBSan: every launch shape of a batch and of one molecule
over sets around its size limits. The leaf orders must equal the reference
QuickSelect's (tests/golden/kd_ref_orders.npz).

A workgroup runs as one host thread per lane, so large sets are slow: sets of up to
1,025 entries by default, up to 8,193 with JAM_EMU_FULL=1."""

import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import golden

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "emu")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or shutil.which("make") is None,
                                reason="needs g++ and make")


def build(target):
    proc = subprocess.run(["make", "-s", "-C", EMU, os.path.join(EMU, "") + "_build/" + target],
                          capture_output=True, text=True)
    if proc.returncode != 0:
        pytest.fail("building the kd emulator failed:\n" + proc.stdout + proc.stderr)
    return os.path.join(EMU, "_build", target)


def run(binary, sets, one_molecule, tmp_path):
    """(leaf orders, error word, launches as (stream, slot, threads))"""
    off = np.concatenate([[0], np.cumsum([len(x) for x in sets])]).astype(np.int64)
    src, dst = tmp_path / "in.bin", tmp_path / "out.bin"
    with open(src, "wb") as f:
        np.array([len(sets), int(one_molecule)], dtype=np.int32).tofile(f)
        off.tofile(f)
        np.concatenate(sets).astype(np.float64).tofile(f)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1", UBSAN_OPTIONS="print_stacktrace=1")
    proc = subprocess.run([binary, str(src), str(dst)], capture_output=True, text=True, env=env, timeout=3600)
    assert proc.returncode == 0, proc.stderr[-4000:]
    out = np.fromfile(dst, dtype=np.int32)
    launches = [tuple(map(int, line.split())) for line in proc.stdout.splitlines()]
    return [out[off[k]:off[k + 1]] for k in range(len(sets))], int(out[-1]), launches


def vectors():
    z = np.load(golden("kd_ref_orders.npz"))
    return z["style"], z["off"], z["q"], z["order"]


def selection(sizes):
    """The sets of these sizes with five distinct coordinates an axis (all of up to
    8,193 entries with JAM_EMU_FULL=1)."""
    style, off, _, _ = vectors()
    n = np.diff(off)
    if os.environ.get("JAM_EMU_FULL") == "1":
        return list(range(len(n)))
    return [i for i in range(len(n)) if int(n[i]) in sizes and style[i] == "int5"]


def check(binary, sel, one_molecule, tmp_path):
    style, off, q, order = vectors()
    sets = [q[off[i]:off[i + 1]].astype(np.float64) / 8.0 for i in sel]
    got, kd_err, launches = run(binary, sets, one_molecule, tmp_path)
    assert kd_err == 0
    bad = [(str(style[i]), len(g)) for i, g in zip(sel, got) if not np.array_equal(g, order[off[i]:off[i + 1]])]
    assert not bad, bad
    return launches


def test_batch(tmp_path):
    launches = check(build("kd_launch_emu"), selection((9, 64, 65, 128, 129, 257, 513, 1025)), False, tmp_path)
    # every kernel but the one-position form of up to 1,024 entries
    assert sorted(slot for _, slot, _ in launches if slot >= 0) == [k for k in range(13) if k != 8]


def test_one_molecule(tmp_path):
    launches = check(build("kd_launch_emu"), selection((9, 65, 513, 1025)), True, tmp_path)
    assert sorted(slot for _, slot, _ in launches if slot >= 0) == [8, 9, 10, 11]


@pytest.mark.parametrize("bound", ["kd_bound_rounds", "kd_bound_jumps"])
@pytest.mark.parametrize("n,one_molecule", [(33, False), (129, True)])
def test_a_bound_that_is_reached_is_reported(tmp_path, bound, n, one_molecule):
    """With bounds too low for any set, the waves that finish small windows (129
    entries) and whole subtrees (33) end and set the error word."""
    _, off, q, _ = vectors()
    i = next(i for i in selection((n,)) if off[i + 1] - off[i] == n)
    _, kd_err, _ = run(build(bound), [q[off[i]:off[i + 1]].astype(np.float64) / 8.0], one_molecule, tmp_path)
    assert kd_err != 0
