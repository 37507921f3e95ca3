"""The pool of device blocks and the staged copies on the CPU, over a HIP runtime
that tests/xfer_host/xfer_host.cpp brings itself: sizes asked of the driver, which
kept block a request takes, what it waits for, and what is freed when.  The HIP headers are
needed, a GPU is not."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime.h")):
        pytest.skip("HIP headers not installed")
    out = str(tmp_path_factory.mktemp("xfer") / "xfer_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "xfer_host", "xfer_host.cpp"), "-lpthread", "-o", out], check=True)
    return out


@pytest.mark.parametrize("check", ["sizes", "card", "devices", "bound", "starve", "copies", "paths"])
def test_pool(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout == f"{check} ok\n"
