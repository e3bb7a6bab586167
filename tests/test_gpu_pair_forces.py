"""Per-atom forces of the full-shell table kernel (csrc/pair_tile.h): no pair
lost or doubled on either side, in every variant of the kernel.

The j side of a cell yields forces only, so pair counts and energies do not
see it.  Here every pair force within the cutoff is between K and 4 K (the
harmonic E = K (r + s)^2 up to 1 nm, s from 0.5 to 0.8 by type pair), and an
atom has at most 300 of them.  FP32 evaluation: r carries the roundings of
three moved coordinates of up to 3 nm (2^-24 each, 1e-7 nm), the chain about 8
more of 2^-24: below 1e-6 of a pair's force from r = 0.2 nm, and below 2e-6
down to the closest pairs at 0.09 nm.  Bound per atom: 3e-6 of the sum of its
pair forces, 300 times less than one pair force.
"""
import itertools

import numpy as np
import pytest

import mdcore as md
import pyoracle as po
import systems

pytestmark = pytest.mark.gpu

K = 0.5
RC = 1.0
# atoms per cell around the matrix tiles of 16 owner atoms (1, 2 tiles with 32
# owner atoms at a time; 2, 3, 4 with 64) and around the owner groups
COUNTS = {32: [0, 1, 4, 15, 16, 17, 31, 32, 33, 40], 64: [1, 16, 32, 33, 47, 48, 49, 63, 64, 65, 97]}


def sites(counts, ncell, h, rng):
    """counts[c] atoms in cell c, on a jittered 5 x 5 x 5 lattice of the cell."""
    x = []
    for c, (i, j, k) in enumerate(itertools.product(*map(range, ncell))):
        s = rng.permutation(125)[:counts[c]]
        p = np.stack([s // 25, s // 5 % 5, s % 5], 1) + 0.5 + rng.uniform(-0.3, 0.3, (len(s), 3))
        x.append((np.array([i, j, k]) + p / 5) * h)
    return np.concatenate(x)


def crowd(r, ntypes, seed, unit=1.0, first=1):
    """Cells of COUNTS[r] atoms, types from `first` up; type pairs share a few
    tables.  The length unit scales everything."""
    rng = np.random.default_rng(seed)
    ncell, h = (3, 4, 5), 1.1
    counts = rng.permutation(np.resize(COUNTS[r], 60))
    assert (counts.mean() > 32) == (r == 64)
    x = sites(counts, ncell, h, rng)
    tabs = [md.harmonic(0.001 * unit, RC * unit, K / unit ** 2, -(0.5 + 0.02 * k) * unit, 1e-3) for k in range(16)]
    ids = range(first, first + ntypes)
    pots = [(i, j, tabs[(i + 3 * j) % 16]) for i in ids for j in ids if i <= j]
    types = rng.integers(first, first + ntypes, len(x)).astype(np.int32)
    return systems.System("crowd", np.zeros(3), np.array(ncell) * h * unit, np.full(3, h * unit), RC * unit, x * unit,
                          types, np.concatenate([[0.0], np.ones(first + ntypes - 1)]), pots)


def pair_force_sums(s, unit):
    """Per atom, at least the sum of its pair forces' magnitudes."""
    out = np.zeros(s.N)
    for a in range(0, s.N, 500):
        d = s.x[a:a + 500, None, :] - s.x[None, :, :]
        d -= np.round(d / s.dim) * s.dim
        r = np.sqrt((d * d).sum(-1)) / unit
        out[a:a + 500] = np.where((r <= RC) & (r > 0), 2 * K * (r + 0.8) / unit, 0.0).sum(1)
    return out


def check_forces(s, flags, proj, unit=1.0):
    o = po.from_system(s).nonbond(po.OR_WINDOW_PROJ if proj else po.OR_WINDOW_REF)
    e = systems.build_engine(s, md.engine_flag_gpu | md.engine_flag_fullshell | flags |
                             (md.engine_flag_projwindow if proj else 0))
    try:
        e.shuffle()
        e.nonbond()
        en = e.energies()
        assert en["pairs"] == o["pairs"]
        bound = 3e-6 * pair_force_sums(s, unit)
        assert bound.max() < K / unit / 300
        err = np.abs(e.forces() - o["f"]).max(1)
        worst = int(np.argmax(err - bound))
        assert np.all(err <= bound), (worst, err[worst], bound[worst])
        assert abs(en["epot_nonbond"] - o["epot"]) <= 1e-6 * o["epot"]
    finally:
        e.close()


# ntypes: the tables' headers and coefficients both fit the kernel's 8 KiB of
# LDS, the headers alone (16 bytes for each of 22 x 22 type pairs), neither
@pytest.mark.parametrize("proj", [False, True])
@pytest.mark.parametrize("flags", [0, md.engine_flag_nosplit])
@pytest.mark.parametrize("ntypes", [2, 21, 24])
@pytest.mark.parametrize("r", [32, 64])
def test_every_pair_on_both_sides(r, ntypes, flags, proj):
    check_forces(crowd(r, ntypes, 100 * r + ntypes), flags, proj)


# cells and cutoff of 1e4 length units, and the null type 0 with potentials
# and atoms of its own: slots without an atom must not count as atoms
@pytest.mark.parametrize("proj", [False, True])
@pytest.mark.parametrize("r", [32, 64])
def test_length_unit_and_type_zero(r, proj):
    check_forces(crowd(r, 2, 7 + r, unit=1e4, first=0), 0, proj, unit=1e4)
