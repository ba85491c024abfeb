"""The walk kernel's layout over cells and LDS (csrc/procell_walk.hpp), which
the host and the device code share, on the CPU (tests/host/walk_checks.cpp,
under AddressSanitizer and UndefinedBehaviorSanitizer)."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def walk_checks(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ is not available")
    exe = str(tmp_path_factory.mktemp("walk") / "walk_checks")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=all", "-I", os.path.join(REPO, "include"),
                        "-I", os.path.join(REPO, "cuda-pro-cell_amd", "csrc"),
                        os.path.join(REPO, "tests", "host", "walk_checks.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]

    def run(check):
        r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 and f"{check}: 0 failed" in r.stdout, r.stdout + r.stderr

    return run


def test_segments_of_any_size(walk_checks):
    walk_checks("segments")


def test_lds_parts_are_aligned(walk_checks):
    walk_checks("lds")
