"""The library's device and pinned memory on a HIP runtime of host memory (native/fake_hip.h): what a
GPU run cannot show without running out of memory, a second device or a launch that fails.  Every
check is one run of native/device_memory.cpp against the built libhv.so."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "highvoronoi.jl_amd")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("device_memory") / "device_memory")
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.check_call([hipcc, "--offload-host-only", "-std=c++17", "-x", "hip", "-I", os.path.join(PKG, "csrc"),
                           os.path.join(ROOT, "tests", "native", "device_memory.cpp"), "-o", exe, "-L", PKG, "-lhv",
                           "-Wl,-rpath," + PKG, "-pthread"])
    return exe


@pytest.mark.parametrize("check", ["failed_export", "queued_work", "released_at_exit", "devices", "idle_given_back",
                                   "integrals_make_room", "staging_taken"])
def test_device_memory(program, check):
    r = subprocess.run([program, check], timeout=120, capture_output=True, text=True,
                       env=dict(os.environ, MALLOC_PERTURB_="90"))   # freed memory is filled
    assert r.returncode == 0, r.stdout + r.stderr
