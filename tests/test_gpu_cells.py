"""The wave-per-cell pair kernel against the cell-per-workgroup kernel, bit for
bit (needs a GPU).  The two differ in the occupancy they are used at only, so
the same particles are run beside fillings that put the mean occupancy on
either side of the line; and against the oracle.  Sizes where the
kernel's stages can go wrong: cells without particles, one home particle, more
than one group turn, cells it leaves to the workgroup (more than 16 home
particles, more than 128 candidates or pairs)."""
import numpy as np
import pytest

import proteinsim2015_amd as ps
from cases import force_params
from helpers import force_rel_err

pytestmark = pytest.mark.gpu

LJ = {"cutOff": 2.5, "kT": 1.0, "wellDepth": 1.0, "yukawaStrength": 0.0, "ljNum": 6,
      "debyeLength": 0.5}
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, seed=1)


def forces(geom, pos, lj=6):
    mods = ps.PLUGINS["LJ"].from_config(ps.Config({**LJ, "ljNum": lj}))
    print(f"n={geom.n} S={geom.cells_per_dim} occupancy={geom.n / geom.ncell:.2f}", flush=True)
    with ps.GpuSystem(geom, mods, INTEG, kernel_path="dense") as s:
        assert s.kernel_info()["path"] == "dense"
        s.set_state(pos)
        st, f = s.forces_now()
    assert st == 0
    return f


@pytest.mark.parametrize("n, S", [(12288, 18), (13000, 16), (12301, 30)])
def test_against_oracle(oracle, n, S):
    geom = ps.SystemGeometry(n=n, box=2.5 * S, cells_per_dim=S, cell_size=2.5, integer=False)
    pos = ps.rsa_positions(n, geom.box, n)
    f = forces(geom, pos)
    sto, fo, _ = oracle.forces(force_params(2, LJ), pos, S, 2.5, geom.box, half_uv=geom.box / 2)
    osum = oracle.pair_stats(force_params(2, LJ), pos, S, 2.5, geom.box, abs_sum=True)[2]
    assert sto == 0
    assert force_rel_err(f, fo, osum).max() <= 1e-6


@pytest.mark.parametrize("lj", [6, 9])
@pytest.mark.parametrize("per_cell", [1.0, 3.0, 5.0, 8.0, 10.0])
def test_same_bits_as_workgroup(per_cell, lj):
    """A fluid block of 7^3 cells in a box of 18^3, once beside 2.6 particles
    per cell (below the line: a wave per cell), once beside 6 (above it: a
    workgroup per cell).  Particles two cells inside the block see the same
    neighbours, in the same cells and the same order."""
    S, b = 18, 7
    box = 2.5 * S
    n = int(per_cell * b ** 3)
    block = ps.rsa_positions(n, 2.5 * b, 5)
    inside = ((block > 5.0) & (block < 2.5 * b - 5.0)).all(1)
    out, occupancy = [], []
    for rest_per_cell in (2.6, 6.0):
        rest = ps.rsa_positions(int(rest_per_cell * S ** 3), box, 6)
        rest = rest[(rest > 2.5 * b + 1.0).any(1) & (rest < box - 1.0).all(1)]
        pos = np.concatenate([block, rest])
        geom = ps.SystemGeometry(n=len(pos), box=box, cells_per_dim=S, cell_size=2.5,
                                 integer=False)
        occupancy.append(geom.n / geom.ncell)
        assert geom.n >= 12288
        out.append(forces(geom, pos, lj)[:n][inside])
    assert occupancy[0] < 3.5 < occupancy[1]
    assert inside.any() and np.array_equal(*out)


def test_crowded_cells():
    """Cells past the wave's limits beside ordinary and empty ones: the forces
    are those of the thread-per-particle kernel to rounding."""
    S, n = 17, 13000
    geom = ps.SystemGeometry(n=n, box=2.5 * S, cells_per_dim=S, cell_size=2.5, integer=False)
    k = np.arange(5)
    tight = 0.5 * np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3) + 5.1
    pos = np.concatenate([tight, ps.rsa_positions(14000, geom.box, 3)])
    keep = np.ones(len(pos), bool)
    keep[125:] = (np.abs(pos[125:] - 6.1) > 2.2).any(1)
    pos = pos[keep][:n]
    mods = ps.PLUGINS["Cal"].from_config(ps.Config({"cutOff": 2.5, "kT": 1.0}))
    out = []
    for path in ("dense", "sparse"):
        with ps.GpuSystem(geom, mods, INTEG, kernel_path=path) as s:
            s.set_state(pos)
            out.append(s.forces_now()[1])
    size = np.abs(out[1]).sum(1)
    near = (np.abs(pos - 6.1) < 6.0).all(1)   # the crowd and what feels it
    assert np.isfinite(out[0]).all()
    assert np.abs(out[0] - out[1])[near].max() <= 1e-10 * size.max()
    assert np.abs(out[0] - out[1])[~near].max() <= 1e-10 * size[~near].max()
