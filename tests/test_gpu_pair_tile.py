"""The full-shell table kernel (csrc/pair_tile.h) and the choices around it,
at the sizes where it can go wrong, against the FP64 oracle.

Tolerances, from the arithmetic: pair counts are exact (FP64 decides the
pairs at the cutoff).  A pair's FP32 force carries r and the Horner chain's
roundings, at most 2^-24 each on r (three coordinates moved by an FP32 shift)
times the steepness of LJ forces (~14) plus ~8 of the chain: 22 x 6e-8 =
1.3e-6 relative in the worst case; 1e-5 of the RMS force leaves room for
sums of opposite forces.  Energies are sums of FP32 pair energies with the
same error, taken into FP64: 1e-5 of the sum of their magnitudes.
"""
import dataclasses

import numpy as np
import pytest

import mdcore as md
import pyoracle as po
import systems

pytestmark = pytest.mark.gpu


def gas(n, box, seed, void=0.0):
    """n atoms at random, 0.28 nm apart at least, argon's table; a void in x."""
    s = systems.argon(4)
    rng = np.random.default_rng(seed)
    x = np.empty((0, 3))
    L = np.array([box * (1.0 - void), box, box])
    while len(x) < n:
        c = rng.random((4 * n, 3)) * L
        for p in c:
            d = np.abs(x - p)
            d = np.minimum(d, box - d)
            if len(x) == 0 or (d * d).sum(1).min() > 0.28 ** 2:
                x = np.vstack([x, p])
                if len(x) == n:
                    break
    return dataclasses.replace(s, dim=np.full(3, box), L=np.full(3, 1.0), x=x, types=np.ones(n, np.int32),
                               v=np.zeros((n, 3)))


def check(s, flags=0, proj=False):
    o = po.from_system(s).nonbond(po.OR_WINDOW_PROJ if proj else po.OR_WINDOW_REF)
    e = systems.build_engine(s, md.engine_flag_gpu | md.engine_flag_fullshell | flags |
                             (md.engine_flag_projwindow if proj else 0))
    e.shuffle()
    e.nonbond()
    f, en = e.forces(), e.energies()
    assert en["pairs"] == o["pairs"]
    rms = np.sqrt((o["f"] ** 2).mean())
    assert np.abs(f - o["f"]).max() <= 1e-5 * np.maximum(rms, np.abs(o["f"]).max())
    assert abs(en["epot_nonbond"] - o["epot"]) <= 1e-5 * (abs(o["epot"]) + 1.0)
    e.nonbond()
    assert np.array_equal(f, e.forces())
    e.close()


# atoms per cell around the tiles of 16, the 32 and 64 owners, the chunk of
# 128 slots (4 cells of 32), with cells that hold none
@pytest.mark.parametrize("proj", [False, True])
@pytest.mark.parametrize("n,box,void", [(27, 3.0, 0.0), (60, 3.0, 0.7), (27 * 15, 3.0, 0.0), (27 * 16, 3.0, 0.0),
                                        (27 * 17, 3.0, 0.0), (27 * 32, 3.3, 0.0), (27 * 33, 3.3, 0.0),
                                        (64 * 9, 4.0, 0.5)])
def test_occupancies(n, box, void, proj):
    check(gas(n, box, n, void), proj=proj)


# one group per owner, and as many as there are
@pytest.mark.parametrize("flags", [0, md.engine_flag_nosplit])
@pytest.mark.parametrize("mk", [lambda: systems.argon(6, jitter=0.05), lambda: systems.mixture(1500, seed=3),
                                lambda: systems.water(300, box=2.4, lattice=(7, 7, 7), cutoff=0.8, cell=0.8),
                                lambda: systems.water(1000, box=3.2, lattice=(10, 10, 10))])
def test_tables_and_windows(mk, flags):
    check(mk(), flags)


# Verlet reuse in resident steps, the half shell's and the surrogate's queues
# included: the steps of engine_step, to the bit
@pytest.mark.parametrize("shell", [md.engine_flag_fullshell, md.engine_flag_halfshell])
def test_verlet_steps_per_shell(shell):
    s = systems.argon(8)
    s.L = np.full(3, 1.12)
    out = []
    for resident in (False, True):
        e = systems.build_engine(s, md.engine_flag_gpu | md.engine_flag_verlet | shell)
        e.setdt(0.002)
        if resident:
            ep = e.gpu_steps(12)[0]
        else:
            ep = []
            for _ in range(12):
                e.step()
                ep.append(e.energies()["epot"])
        out.append((np.array(ep), e.positions(), e.forces()))
        e.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
