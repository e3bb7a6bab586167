"""A pass that fails must leave the next one its work: the half shell's and
the surrogate's kernels take their cells from queues that a pass's totals
clear, so a pass that ends in an error before them leaves the queues used up.
tests/csrc/pass_error_check.cpp runs the built library's host code on stubs
of the HIP runtime (no GPU) and fails a launch and an event."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mdcore-history_amd"
HIP = Path("/opt/rocm/include/hip/hip_runtime_api.h")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_pass_after_a_failed_one_has_work(tmp_path):
    exe = tmp_path / "pass_error_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", f"-I{HIP.parents[1]}",
                    f"-I{ROOT / 'include'}", "-o", str(exe), str(ROOT / "tests" / "csrc" / "pass_error_check.cpp"),
                    "-rdynamic", f"-L{PKG / 'lib'}", "-lmdcore_gpu", f"-Wl,-rpath,{PKG / 'lib'}",
                    f"-L{HIP.parents[2] / 'lib'}", f"-Wl,-rpath-link,{HIP.parents[2] / 'lib'}"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
