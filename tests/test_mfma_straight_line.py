"""The compiled pair kernels read an MFMA's result in the straight-line code
after it: the compiler puts the wait states that the read needs between the two,
and has left them out across a branch.  Reads the assembly of this build's own
source."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / "mdcore-history_amd"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def registers(operands):
    out = set()
    for a, b, c in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", operands):
        out |= {int(c)} if c else set(range(int(a), int(b) + 1))
    return out


def branches_before_the_read(asm):
    """(MFMAs, those with a label or branch before an instruction that names
    the result)."""
    lines = [t for t in (l.split(";")[0].strip() for l in asm.split("\n")) if t and (t.endswith(":") or t[0] != ".")]
    n, bad = 0, []
    for i, l in enumerate(lines):
        if not l.startswith("v_mfma"):
            continue
        n += 1
        dest = registers(l.split(None, 1)[1].split(",")[0])
        for t in lines[i + 1:]:
            if t.endswith(":") or t.startswith(("s_cbranch", "s_branch", "s_endpgm", "s_setpc")):
                bad.append(l)
                break
            if dest & registers(t.partition(" ")[2] or t.partition("\t")[2]):
                break
    return n, bad


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_results_are_read_without_a_branch(tmp_path):
    make = subprocess.run(["make", "-n", "-B", "-C", str(PKG)], capture_output=True, text=True, check=True).stdout
    line = next(l for l in make.split("\n") if "-c" in l.split() and "engine_gpu.hip" in l)
    asm = tmp_path / "engine_gpu.s"
    cmd = line.split()
    cmd = cmd[:cmd.index("-c")] + ["--cuda-device-only", "-S", cmd[cmd.index("-c") + 1], "-o", str(asm)]
    subprocess.run(cmd, check=True, capture_output=True)
    n, bad = branches_before_the_read(asm.read_text())
    assert n > 0 and not bad, (n, bad)


def test_a_branch_is_found():
    mfma = "\tv_mfma_f32_16x16x4_f32 v[4:7], v1, v2, v[4:7]\n"
    assert branches_before_the_read(mfma + "\ts_nop 9\n\tv_add_f32_e32 v0, v5, v1\n") == (1, [])
    assert len(branches_before_the_read(mfma + "\ts_cbranch_scc0 .LBB0_1\n\tv_add_f32_e32 v0, v5, v1\n")[1]) == 1
    assert len(branches_before_the_read(mfma + ".LBB0_1:\n\tv_add_f32_e32 v0, v5, v1\n")[1]) == 1
