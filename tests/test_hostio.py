"""The kept buffers and copies of the host-array calls (lenstool-hpc_amd/csrc/lt_hostio.cpp) where memory runs out or is
refused and where copies fail, on the CPU with a stand-in for the HIP runtime (tests/cpp/fake_hip)."""
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostio") / "hostio_check")
    csrc = os.path.join(ROOT, "lenstool-hpc_amd", "csrc")
    cpp = os.path.join(ROOT, "tests", "cpp")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-I" + os.path.join(cpp, "fake_hip"), "-I" + csrc,
                    "-I" + os.path.join(ROOT, "include"), os.path.join(cpp, "hostio_check.cpp"),
                    os.path.join(csrc, "lt_hostio.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["room", "pinned", "errors"])
def test_hostio(check, what):
    r = subprocess.run([check, what], capture_output=True, text=True, timeout=60)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK")
