"""The output bin set's values and the bin of every (row, generation) against
their definition (tests/host/bin_checks.cpp, under AddressSanitizer and
UndefinedBehaviorSanitizer): shared mantissas, phi equal to a value, at and
below the smallest normal number, rows below phi and negative ones."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "cuda-pro-cell_amd", "csrc")


def test_bins_and_their_entries(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ is not available")
    exe = str(tmp_path / "bin_checks")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=all", "-I", os.path.join(REPO, "include"), "-I", CSRC,
                        os.path.join(REPO, "tests", "host", "bin_checks.cpp"), os.path.join(CSRC, "procell_setup.cpp"),
                        "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and " 0 failed" in r.stdout, r.stdout + r.stderr
