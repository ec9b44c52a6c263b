"""The thread-per-particle gather at the sizes where its stages can go wrong
(needs a GPU): waves with idle lanes and systems below one wave, candidate
columns that overflow (21 rows) and rounds that overflow (128 pairs per wave),
one and four lanes per particle, particles on the box faces and on cell
boundaries.  Neighbour sets must equal the oracle's exactly; forces are held
to the parity tolerance (1e-6 relative, |dF_i| / max(|F_i|, sum_j |f_ij|))."""
import numpy as np
import pytest

import proteinsim2015_amd as ps
from cases import PHI_P_C2, force_params
from helpers import force_rel_err

pytestmark = pytest.mark.gpu

AO = {"cutOff": 1.1, "kT": 1.0, "wellDepth": PHI_P_C2}
LJ = {"cutOff": 2.5, "kT": 1.0, "wellDepth": 1.0, "yukawaStrength": 0.0, "ljNum": 6,
      "debyeLength": 0.5}
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-3, seed=1)


def check(oracle, plugin, mask, cfg, geom, pos):
    fp = force_params(mask, cfg)
    mods = ps.PLUGINS[plugin].from_config(ps.Config(cfg))
    S, cell, L = geom.cells_per_dim, geom.cell_size, geom.box
    print(f"{plugin} n={geom.n} S={S} occupancy={geom.n / S ** 3:.2f}", flush=True)
    ocnt, ohs, osum = oracle.pair_stats(fp, pos, S, cell, L, abs_sum=True)
    sto, fo, _ = oracle.forces(fp, pos, S, cell, L, half_uv=L / 2)
    with ps.GpuSystem(geom, mods, INTEG, kernel_path="sparse") as sysg:
        sysg.set_state(pos)
        cnt, hs = sysg.pair_stats()
        st, f = sysg.forces_now()
    assert sto == 0 and st == 0
    assert np.array_equal(cnt, ocnt) and np.array_equal(hs, ohs)
    assert force_rel_err(f, fo, osum).max() <= 1e-6
    return cnt


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 1001])
def test_partial_waves(oracle, n):
    geom = ps.SystemGeometry(n=n, box=24.2, cells_per_dim=22, cell_size=1.1, integer=False)
    check(oracle, "AO", 4, AO, geom, ps.rsa_positions(n, geom.box, 40 + n))


@pytest.mark.parametrize("cells, phi", [(6, 0.30), (5, 0.10), (4, 0.20)])
def test_columns_and_rounds_overflow(oracle, cells, phi):
    """Cells of the cutoff and coarser: 80 to 400 candidates per particle."""
    box = 6 * 2.6
    n = int(phi * box ** 3 / 0.5236)
    geom = ps.SystemGeometry(n=n, box=box, cells_per_dim=cells,
                             cell_size=box / cells, integer=False)
    cnt = check(oracle, "LJ", 2, LJ, geom, ps.rsa_positions(n, box, 7))
    assert cnt.sum() > 0


def test_one_lane_per_particle_overflows(oracle):
    """262,144 particles of an LJ system at three per cell: one lane each."""
    n = 262144
    geom = ps.SystemGeometry.exact(n, 0.10, 2.5)
    check(oracle, "LJ", 2, LJ, geom, ps.rsa_positions(n, geom.box, 11))


def test_faces_and_cell_boundaries(oracle):
    """A lattice with sites exactly on the faces (0 and the last double below
    L) and on cell boundaries, all pairs across the periodic faces present."""
    S, cell = 8, 1.25
    L = S * cell
    g = np.arange(S) * cell
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    pos[pos[:, 2] == 0.0, 0] += 0.1
    pos[::7] = np.where(pos[::7] == 0.0, np.nextafter(L, 0), pos[::7])
    geom = ps.SystemGeometry(n=len(pos), box=L, cells_per_dim=S, cell_size=cell, integer=False)
    cfg = dict(AO, cutOff=1.25)
    cnt = check(oracle, "AO", 4, cfg, geom, np.ascontiguousarray(pos))
    assert cnt.max() >= 1
