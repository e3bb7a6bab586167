"""Sums of the full-shell table kernel (csrc/pair_tile.h): an atom's forces add
up in FP64, so that small ones beside large ones that cancel are not lost.

Atoms A and S are two lattices, each A an inversion centre of the S: the 32 S
within the cutoff pull it with forces of about 2^20 each, which cancel.  Their
coordinates are multiples of 2^-7 nm, so that opposite S have the same FP32
distance and force bits and their exact products cancel exactly.  Atoms W at
random sites pull with forces of about 1.  A's force is the sum of its W's,
each within 3e-6 of itself (the FP32 evaluation, as in
test_gpu_pair_forces.py), and what FP64 sums of 2^20 x 32 lose, 2^-28 for each
of at most 100 additions.  A single sum of S and W forces in FP32 loses 2^-4.
"""
import itertools

import numpy as np
import pytest

import mdcore as md
import pyoracle as po
import systems

pytestmark = pytest.mark.gpu

RC = 1.0
H = 1.125  # cell
K = 0.5    # E = K (r + 0.5)^2


def lattice(ncell, shift):
    """2 x 2 x 2 sites per cell."""
    g = np.array(list(itertools.product(range(2 * ncell), repeat=3)), float)
    return (g + shift) * (H / 2)


def crystal(nw, ncell=4, seed=5):
    """Cells of 8 A (type 1), 8 S (type 2) and about nw W (type 3)."""
    rng = np.random.default_rng(seed)
    a, s = lattice(ncell, 0.25), lattice(ncell, 0.75)
    w = rng.random((nw * ncell ** 3, 3)) * ncell * H
    d = np.abs(w[:, None, :] - a[None, :, :])
    d = np.minimum(d, ncell * H - d)
    w = w[(d * d).sum(-1).min(1) > 0.01]
    x = np.concatenate([a, s, w])
    types = np.repeat([1, 2, 3], [len(a), len(s), len(w)]).astype(np.int32)
    strong = md.harmonic(0.001, RC, K * 2.0 ** 20, -0.5, 1e-3)
    weak = md.harmonic(0.001, RC, K, -0.5, 1e-3)
    return systems.System("crystal", np.zeros(3), np.full(3, ncell * H), np.full(3, H), RC, x, types,
                          np.array([0.0, 1.0, 1.0, 1.0]), [(1, 2, strong), (1, 3, weak)])


# 16 and 46 atoms per cell: 32 and 64 owner atoms at a time; one group per
# owner and as many as there are
@pytest.mark.parametrize("proj", [False, True])
@pytest.mark.parametrize("flags", [0, md.engine_flag_nosplit])
@pytest.mark.parametrize("nw", [4, 30])
def test_large_forces_that_cancel(nw, flags, proj):
    s = crystal(nw)
    na = int((s.types == 1).sum())
    o = po.from_system(s).nonbond(po.OR_WINDOW_PROJ if proj else po.OR_WINDOW_REF)
    d = s.x[:na, None, :] - s.x[None, s.types == 3, :]
    d -= np.round(d / s.dim) * s.dim
    r = np.sqrt((d * d).sum(-1))
    weak = np.where(r <= RC, 2 * K * (r + 0.5), 0.0).sum(1)
    assert np.abs(o["f"][:na]).max() < weak.max()  # the S cancel
    e = systems.build_engine(s, md.engine_flag_gpu | md.engine_flag_fullshell | flags |
                             (md.engine_flag_projwindow if proj else 0))
    try:
        e.shuffle()
        e.nonbond()
        assert e.energies()["pairs"] == o["pairs"]
        err = np.abs(e.forces() - o["f"])[:na].max(1)
        assert np.all(err <= 3e-6 * weak + 100 * 2.0 ** -28), (err / weak).max()
    finally:
        e.close()
