"""A pass after one that ended in an error between its upload and its end does
not write the pinned block that the first one's copy may still read: the two
would mix, and a kernel takes indices from the block.
tests/csrc/stage_reuse_check.cpp runs the built library's host code on stubs of
the HIP runtime (no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mdcore-history_amd"
HIP = Path("/opt/rocm/include/hip/hip_runtime_api.h")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_upload_waits_for_the_copy_before(tmp_path):
    exe = tmp_path / "stage_reuse_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", f"-I{HIP.parents[1]}",
                    f"-I{ROOT / 'include'}", "-o", str(exe), str(ROOT / "tests" / "csrc" / "stage_reuse_check.cpp"),
                    "-rdynamic", f"-L{PKG / 'lib'}", "-lmdcore_gpu", f"-Wl,-rpath,{PKG / 'lib'}",
                    f"-L{HIP.parents[2] / 'lib'}", f"-Wl,-rpath-link,{HIP.parents[2] / 'lib'}"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
