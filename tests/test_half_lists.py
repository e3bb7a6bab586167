"""The half shell's neighbour lists and force slots follow the order of the
tasks, in which k_fold adds a cell's forces up.  tests/csrc/half_list_check.cpp
reads what the built library hands its kernels, on stubs of the HIP runtime
(no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mdcore-history_amd"
HIP = Path("/opt/rocm/include/hip/hip_runtime_api.h")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_half_lists_in_task_order(tmp_path):
    exe = tmp_path / "half_list_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", f"-I{HIP.parents[1]}",
                    f"-I{ROOT / 'include'}", "-o", str(exe), str(ROOT / "tests" / "csrc" / "half_list_check.cpp"),
                    "-rdynamic", f"-L{PKG / 'lib'}", "-lmdcore_gpu", f"-Wl,-rpath,{PKG / 'lib'}",
                    f"-L{HIP.parents[2] / 'lib'}", f"-Wl,-rpath-link,{HIP.parents[2] / 'lib'}"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
