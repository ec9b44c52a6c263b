"""Neighbour sets of the wave-per-cell pair kernel against the oracle's brute
force (needs a GPU), at densities and sizes that context runs it at: counts and
partner-hash sums are whole numbers and must be equal.  Cells without
particles, cells it leaves to the workgroup, and a lattice whose neighbours lie
exactly on the cutoff (the strict r^2 < rc^2 has them outside)."""
import numpy as np
import pytest

import proteinsim2015_amd as ps
from cases import force_params

pytestmark = pytest.mark.gpu

CFG = {"cutOff": 2.5, "kT": 1.0}
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, seed=1)


def check(oracle, pos, S, path="auto"):
    g = ps.SystemGeometry(n=len(pos), box=2.5 * S, cells_per_dim=S, cell_size=2.5, integer=False)
    print(f"n={g.n} S={S} occupancy={g.n / g.ncell:.2f}", flush=True)
    assert g.n >= 12288 and g.n / g.ncell < 3.5
    ocnt, ohs = oracle.pair_stats(force_params(1, CFG), pos, S, 2.5, g.box)[:2]
    with ps.GpuSystem(g, ps.Calibration(cutoff=2.5), INTEG, kernel_path=path) as s:
        assert s.kernel_info()["path"] == "dense"
        s.set_state(pos)
        cnt, hs = s.pair_stats()
    assert np.array_equal(cnt, ocnt) and np.array_equal(hs, ohs)
    return cnt


@pytest.mark.parametrize("n, S, path", [(12288, 18, "auto"), (13000, 16, "auto"),
                                        (30011, 21, "auto"), (12301, 30, "dense")])
def test_fluid(oracle, n, S, path):
    assert check(oracle, ps.rsa_positions(n, 2.5 * S, n), S, path).max() > 0


def test_cells_left_to_the_workgroup(oracle):
    S = 17
    k = np.arange(6)
    tight = 1.0 * np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3) + 5.1
    rest = ps.rsa_positions(14000, 2.5 * S, 3)
    rest = rest[(np.abs(rest - 7.6) > 3.6).any(1)]
    assert check(oracle, np.concatenate([tight, rest]), S).max() > 40


def test_neighbours_on_the_cutoff(oracle):
    """A third of the sites of a lattice with spacing 1.25 = rc / 2."""
    S = 18
    k = np.arange(2 * S) * 1.25 + 0.5
    pos = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)
    check(oracle, pos[np.random.default_rng(2).permutation(len(pos))[:15552]], S)
