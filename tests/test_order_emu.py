"""The order of the atoms of molecules whose serial numbers descend at a few
atoms (k_run_order in pyjess_amd/csrc/jam_ingest.h), run on the CPU under the
emulation of tests/emu/ with AddressSanitizer and UBSan, at the start of a batch
and at the end of one of 2^31 - 1 atoms."""

import shutil
import subprocess

import pytest

from tests.test_kd_launch_emu import build

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or shutil.which("make") is None,
                                reason="needs g++ and make")


@pytest.mark.parametrize("before", [0, 255, 1 << 30, (1 << 31) - 1 - 1000])
def test_order(before):
    proc = subprocess.run([build("order_emu"), str(before)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout + proc.stderr[-4000:]
    assert proc.stdout == "4 descents\n"
