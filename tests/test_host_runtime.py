"""The library's host code on the CPU (tests/drivers/host_runtime.cpp): its contexts,
graphs, tiles and batch engine against a runtime and kernels that keep only their
bookkeeping."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.environ.get("ROCM_PATH", "/opt/rocm")

CHECKS = ["geometry_failure", "mask_attribute", "graph_start", "autotune_start", "autotune_own_tile",
          "batch_open_rows", "batch_waiting", "persistent_grid"]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None or not os.path.isfile(os.path.join(HIP, "include", "hip", "hip_runtime.h")):
        pytest.skip("no C++ compiler or HIP headers")
    exe = str(tmp_path_factory.mktemp("host") / "host_runtime")
    csrc = os.path.join(ROOT, "ibtfo_amd", "csrc")
    subprocess.run([cxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(HIP, "include"), "-o", exe,
                    os.path.join(ROOT, "tests", "drivers", "host_runtime.cpp"), os.path.join(csrc, "ibtfo_capi.cpp"),
                    os.path.join(csrc, "ibtfo_batch.cpp"), "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("check", CHECKS)
def test_host_runtime(driver, check):
    r = subprocess.run([driver, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
