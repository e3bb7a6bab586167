"""Energies of the projected window do not depend on the number of compute
units: the rule that rounds its pairs goes by the number of cells.
tests/csrc/cu_count_check.cpp runs the built library's host code on stubs of
the HIP runtime (no GPU)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mdcore-history_amd"
HIP = Path("/opt/rocm/include/hip/hip_runtime_api.h")


@pytest.mark.skipif(shutil.which("g++") is None or not HIP.exists(), reason="needs g++ and the HIP headers")
def test_rounding_rule_without_the_device(tmp_path):
    exe = tmp_path / "cu_count_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-w", f"-I{HIP.parents[1]}",
                    f"-I{ROOT / 'include'}", "-o", str(exe), str(ROOT / "tests" / "csrc" / "cu_count_check.cpp"),
                    "-rdynamic", f"-L{PKG / 'lib'}", "-lmdcore_gpu", f"-Wl,-rpath,{PKG / 'lib'}",
                    f"-L{HIP.parents[2] / 'lib'}", f"-Wl,-rpath-link,{HIP.parents[2] / 'lib'}"], check=True)

    def cap(cus, edge):
        r = subprocess.run([str(exe), str(cus), str(edge)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
        return int(r.stdout)

    # 25^3 and 26^3 cells lie on both sides of 16,384
    for edge, want in ((10, 32), (25, 32), (26, 28), (30, 28)):
        assert [cap(cus, edge) for cus in (64, 256, 304)] == [want] * 3
