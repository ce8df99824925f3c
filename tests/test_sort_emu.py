"""The kernels that order complete matches by groups of level-0 rows, run on the
CPU under the emulation of tests/emu/ with AddressSanitizer and UBSan, against
a comparison sort: ranking of all groups, the LDS sort, and listed large
groups (more than 512 matches: the emulation's tiles are a quarter of the
device's); one and several rows to a group, templates of one atom, one match,
and keys of several 64-bit words that begin alike."""

import os
import shutil
import subprocess

import pytest

from tests.test_kd_launch_emu import build

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or shutil.which("make") is None,
                                reason="needs g++ and make")

CASES = [
    # molecules, entries, rows, matches to a row, shift, way, template sizes;
    # then: at least as many matches in the largest group, words, matches
    # that share their first word
    ((2, 40, 60, 20, 0, "ranked", 4, 1, 6, 3), 10, 1, 0),
    ((2, 40, 60, 20, 3, "tiled", 4, 1, 6, 3), 20, 1, 0),
    ((1, 100, 60, 1, 2, "ranked", 1), 2, 1, 0),
    ((1, 100, 60, 1, 5, "tiled", 1), 2, 1, 0),
    ((1, 10, 1, 1, 0, "ranked", 2), 1, 1, 0),
    ((1, 10, 1, 1, 0, "tiled", 2), 1, 1, 0),
    ((3, 6000, 9, 70, 0, "ranked", 24, 2, 12), 70, 5, 50),
    ((3, 6000, 9, 70, 4, "tiled", 24, 1, 12), 70, 5, 50),
    ((1, 2000, 3, 700, 0, "tiled", 15, 13), 513, 3, 300),
    ((1, 2000, 3, 700, 2, "tiled", 15, 13), 513, 3, 300),
]


@pytest.mark.parametrize("case,group,words,shared", CASES, ids=["-".join(map(str, c[0])) for c in CASES])
def test_order(case, group, words, shared):
    proc = subprocess.run([build("sort_emu"), "7", *map(str, case)], capture_output=True, text=True, timeout=600,
                          env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1"))
    assert proc.returncode == 0, proc.stdout + proc.stderr[-4000:]
    got = list(map(int, proc.stdout.split()))
    print(got)
    assert got[1] >= group and got[2] >= words and got[3] >= shared
