"""A forked child reads positions, velocities and forces out, as a program's
worker processes do, although the parent's loops ran with several threads (which
the child does not have)."""
import os
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

PROGRAM = """
import os, signal
import numpy as np
import mdcore as md
import systems

s = systems.argon(18)
e = systems.build_engine(s, md.engine_flag_gpu, start=False)
e.shuffle()
x = e.positions()
assert s.N >= 16384
pid = os.fork()
if pid == 0:
    signal.alarm(20)
    e.shuffle()
    same = np.array_equal(x, e.positions()) and len(e.velocities()) == len(e.forces()) == s.N
    os._exit(0 if same else 1)
status = os.waitpid(pid, 0)[1]
assert np.array_equal(x, e.positions())
raise SystemExit(0 if status == 0 else f"child ended with status {status}")
"""


def test_getters_in_a_forked_child():
    path = os.pathsep.join([str(ROOT / "mdcore-history_amd"), os.environ.get("PYTHONPATH", "")])
    r = subprocess.run([sys.executable, "-c", PROGRAM], capture_output=True, text=True, timeout=90,
                       env=dict(os.environ, PYTHONPATH=path, OMP_NUM_THREADS="8"))
    assert r.returncode == 0, r.stderr
