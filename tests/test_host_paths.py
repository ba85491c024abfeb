"""libprocell's host code on the CPU: the built library over a stand-in for
the HIP runtime (tests/host/fake_hip.cpp), driven by tests/host/host_paths.cpp
through the C ABI.  Kernels are recorded and not run; device memory is host
memory."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "cuda-pro-cell_amd", "csrc")
BUILD = os.path.join(REPO, "cuda-pro-cell_amd", "_build")
HOST = os.path.join(REPO, "tests", "host")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def host_paths(procell_lib, tmp_path_factory):
    if not shutil.which("g++") or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("g++ or the HIP headers are not available")
    out = tmp_path_factory.mktemp("host")
    fake, exe = str(out / "libamdhip64.so.7"), str(out / "host_paths")
    flags = ["-std=c++17", "-O1", "-g", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__",
             "-I", os.path.join(ROCM, "include"), "-I", os.path.join(REPO, "include"), "-I", CSRC]
    for cmd in (["g++", *flags, "-fPIC", "-shared", "-Wl,-soname,libamdhip64.so.7",
                 os.path.join(HOST, "fake_hip.cpp"), "-o", fake],
                ["g++", *flags, os.path.join(HOST, "host_paths.cpp"), "-o", exe, "-L", BUILD, "-lprocell", fake,
                 f"-Wl,-rpath,{BUILD}", "-Wl,--unresolved-symbols=ignore-in-shared-libs"]):
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-4000:]

    def run(check):
        env = dict(os.environ, LD_LIBRARY_PATH=str(out))
        r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120, env=env)
        assert r.returncode == 0 and f"{check}: 0 failed" in r.stdout, r.stdout + r.stderr

    return run


def test_results_after_a_run_that_failed_late(host_paths):
    host_paths("stage")


def test_rows_that_fit_the_static_scratch(host_paths):
    host_paths("noalloc")


def test_calls_around_a_device_reset(host_paths):
    host_paths("reset")


def test_kernel_of_a_run(host_paths):
    host_paths("kernel")


def test_tally_window_of_deep_rows(host_paths):
    host_paths("window")


def test_autotuner_times_each_layout_once(host_paths):
    host_paths("autotune")


def test_relaxed_plans_of_many_sets_bound_their_stacks(host_paths):
    host_paths("stacks")
