"""The delensing scan's tile test (lenstool-hpc_amd/csrc/lt_delense_tile.h) on the host, compiled from the same
header as the device kernel: no source that it skips for a tile has a hit in one of the tile's cells. Host
only; the device kernel's results are compared with the oracle bit for bit by the delensing GPU tests."""
import os
import subprocess

import pytest

from conftest import ROOT
from test_delense_cull import HIPCC


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_tile_test_is_sound(tmp_path):
    exe = tmp_path / "delense_tile_check"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "lenstool-hpc_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "delense_tile_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe), "40000"], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr
