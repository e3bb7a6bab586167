"""Resident steps whose next pass, launched before the migration's outcome is
known, has to be done over: a cell grows past the launch's margin (4 atoms and
an eighth, not past the sort's variants at 64 and 480), or a particle crosses
more than one cell in a step.  The steps are engine_step's, bit for bit; that
both happened is read off the host-driven run."""
import itertools

import numpy as np
import pytest

import mdcore as md
import surrogate as sg
import systems

pytestmark = pytest.mark.gpu

DT = 0.01


def slab(n0, ncell, seed=3):
    """n0 atoms per cell of 1 nm at rest; those of cell layer 1 move by 0.9
    cells a step along x, so that layer 2 holds twice as many after the first;
    four others by 2.3 cells along y."""
    rng = np.random.default_rng(seed)
    cells = np.array(list(itertools.product(*map(range, ncell))), float)
    x = (cells[:, None, :] + 0.15 + 0.7 * rng.random((len(cells), n0, 3))).reshape(-1, 3)
    layer = np.repeat(cells[:, 0], n0)
    v = np.zeros_like(x)
    v[layer == 1, 0] = 0.9 / DT
    v[np.flatnonzero(layer == 3)[:4], 1] = 2.3 / DT
    pot = md.harmonic(0.001, 1.0, 0.5 / n0, 0.5, 1e-3)
    return systems.System("slab", np.zeros(3), np.array(ncell, float), np.full(3, 1.0), 1.0, x,
                          np.ones(len(x), np.int32), np.array([0.0, 1.0]), [(1, 1, pot)], v=v)


def margin(n):
    lim = n + 4 + n // 8
    for m in (64, 480):
        lim = m if n <= m < lim else lim
    return lim


# 8 and 20 atoms per cell; to the sort's limits of 64 and 480 and past them
@pytest.mark.parametrize("flags", [0, md.engine_flag_nosplit])
@pytest.mark.parametrize("n0,ncell", [(8, (6, 5, 7)), (20, (6, 6, 6)), (60, (5, 5, 5)), (470, (4, 3, 3))])
def test_pass_done_over(n0, ncell, flags):
    s, n, nc = slab(n0, ncell), 4, int(np.prod(ncell))
    out, grown, far = [], [], []
    for resident in (False, True):
        e = systems.build_engine(s, md.engine_flag_gpu | md.engine_flag_fullshell | flags)
        try:
            e.setdt(DT)
            if resident:
                ep = e.gpu_steps(n)[0]
            else:
                ep = []
                big = n0
                for k in range(n):
                    e.step()
                    now = int(e.cells(nc)[0].max())
                    if k + 1 < n:  # a pass followed
                        grown.append(now > margin(big))
                        # past the neighbour cell
                        far.append(np.abs(e.velocities()).max() * DT > 2.0)
                    big = now
                    ep.append(e.energies()["epot"])
            c, ids = e.cells(nc)
            out.append((np.array(ep), c, ids, e.positions(), e.velocities(), e.forces()))
            assert np.all(np.isfinite(out[-1][0]))
        finally:
            e.close()
    assert any(grown) and any(far)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_verlet_steps_surrogate():
    """Sort reuse in resident steps of the surrogate (its work queues)."""
    s = systems.argon(8)
    s.L = np.full(3, 1.12)
    out = []
    for resident in (False, True):
        e = systems.build_engine(s, md.engine_flag_gpu | md.engine_flag_verlet)
        try:
            e.mlp_init(*sg.pair_domains(e, s), seed=4)
            e.setflags(md.engine_flag_mlp, 0)
            e.setdt(0.0005)
            if resident:
                ep = e.gpu_steps(12)[0]
            else:
                ep = []
                for _ in range(12):
                    e.step()
                    ep.append(e.energies()["epot"])
            out.append((np.array(ep), e.positions(), e.forces()))
            assert np.all(np.isfinite(out[-1][0]))
        finally:
            e.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
