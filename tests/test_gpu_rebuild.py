"""The cell rebuild at the sizes where its stages can go wrong (needs a GPU):
one, two and four particles per lane, a last tile that is not whole, tiles
without particles, more tiles than a workgroup sums itself, cells past their
bin's row (chains) and tiles past the LDS list.  The start table and the slot
order are whole numbers and must equal a stable counting sort exactly, from a
fresh state and after steps (order within a cell = previous slot order)."""
import numpy as np
import pytest

import proteinsim2015_amd as ps

pytestmark = pytest.mark.gpu

AO = ps.AOPotential(kT=1.0, well_depth=ps.AOPotential.well_depth_for_contact(3.0, 0.1),
                    cutoff=1.1)
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-3, seed=3)


def keys(pos, g):
    c = np.minimum((pos / g.cell_size).astype(np.int64), g.cells_per_dim - 1)
    return c[:, 0] + g.cells_per_dim * (c[:, 1] + g.cells_per_dim * c[:, 2])


def check(sysg, g, before):
    """The table and order now against a stable sort of the order before."""
    _, start, ids = sysg.cells()
    k = keys(sysg.get_state()["pos"], g)
    want = before[np.argsort(k[before], kind="stable")]
    assert np.array_equal(np.asarray(ids), want)
    assert np.array_equal(np.asarray(start),
                          np.concatenate([[0], np.cumsum(np.bincount(k, minlength=g.ncell))]))
    return want


@pytest.mark.parametrize("n, S", [(1, 4), (63, 5), (1000, 22), (4097, 9), (32768, 31),
                                  (131071, 70), (131072, 70), (300007, 96), (1048576, 90),
                                  (2000, 212)])
def test_order_and_starts(n, S):
    g = ps.SystemGeometry(n=n, box=1.2 * S, cells_per_dim=S, cell_size=1.2, integer=False)
    pos = np.random.default_rng(n).uniform(0, g.box, (n, 3))
    with ps.GpuSystem(g, [AO], INTEG) as sysg:
        sysg.set_state(pos)
        check(sysg, g, np.arange(n))


@pytest.mark.parametrize("n, S", [(1500, 12), (40001, 36), (140001, 54), (1100003, 106)])
def test_order_after_steps(n, S):
    g = ps.SystemGeometry(n=n, box=1.2 * S, cells_per_dim=S, cell_size=1.2, integer=False)
    m = int(np.ceil(n ** (1 / 3)))   # a lattice: no overlaps
    k = (np.arange(m) + 0.5) * (g.box / m)
    pos = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)[:n]
    with ps.GpuSystem(g, [AO], INTEG) as sysg:
        sysg.set_state(pos)
        order = check(sysg, g, np.arange(n))
        for _ in range(3):
            assert sysg.step(1) == 0
            order = check(sysg, g, order)


@pytest.mark.parametrize("n, S, crowd", [(300, 8, 300), (5000, 16, 700), (5000, 16, 5000),
                                         (140000, 60, 3000)])
def test_crowded_cells(n, S, crowd):
    """crowd particles in two cells, the rest anywhere; then a second state,
    so that what the first left in the bins would show."""
    g = ps.SystemGeometry(n=n, box=1.2 * S, cells_per_dim=S, cell_size=1.2, integer=False)
    rng = np.random.default_rng(crowd)
    pos = rng.uniform(0, g.box, (n, 3))
    pos[rng.permutation(n)[:crowd]] = rng.uniform(0, 1.2, (crowd, 3)) * [2, 1, 1] + 2.4
    with ps.GpuSystem(g, [AO], INTEG) as sysg:
        for p in (pos, pos[::-1].copy(), rng.uniform(0, g.box, (n, 3))):
            sysg.set_state(p)
            check(sysg, g, np.arange(n))
