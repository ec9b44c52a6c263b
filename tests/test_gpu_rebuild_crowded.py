"""The cell rebuild where cells are crowded or nearly all empty (needs a GPU), from
step to step, so that whatever one rebuild leaves behind shows in the next:
mean occupancies on both sides of the line of the split rebuild for one, two and
four particles per lane; dense spots in a dilute box (tiles done in batches,
cells past their bin as chains, cells past the list in LDS); tiles of 2048 cells
and more tiles than a workgroup sums itself.  The order is whole numbers and
must equal a stable counting sort of the order before."""
import numpy as np
import pytest

import proteinsim2015_amd as ps

pytestmark = pytest.mark.gpu

# no forces (wellDepth 0): only the order is looked at, and particles that come
# close are no error here
FREE = ps.LennardJones(kT=1.0, well_depth=0.0, yukawa_strength=0.0, lj_num=6, cutoff=0.05)
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=0.05, seed=3)


def lattice(n, width):
    m = int(np.ceil(n ** (1 / 3) - 1e-9))
    k = (np.arange(m) + 0.5) * (width / m)
    return np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)[:n]


def follow(n, S, pos, steps=3, path="auto"):
    """Order and start table after set_state and after each step."""
    g = ps.SystemGeometry(n=n, box=1.2 * S, cells_per_dim=S, cell_size=1.2, integer=False)
    print(f"n={n} S={S} occupancy={n / g.ncell:.3f}", flush=True)
    moved = 0
    with ps.GpuSystem(g, FREE, INTEG, kernel_path=path) as s:
        s.set_state(pos)
        before, old = np.arange(n), None
        for k in range(steps + 1):
            if k:
                assert s.step(1) in (0, ps.ERR_OVERLAP)
            _, start, ids = s.cells()
            x = s.get_state()["pos"]
            c = np.minimum((x / g.cell_size).astype(np.int64), S - 1)
            key = c[:, 0] + S * (c[:, 1] + S * c[:, 2])
            want = before[np.argsort(key[before], kind="stable")]
            assert np.array_equal(ids, want)
            assert np.array_equal(start[1:], np.cumsum(np.bincount(key, minlength=g.ncell)))
            moved += 0 if old is None else (key != old).sum()
            before, old = want, key
    assert moved > 0 or steps == 0


@pytest.mark.parametrize("n, S", [(3600, 4), (3800, 4), (10000, 4), (30011, 4), (24800, 6),
                                  (140000, 11), (140000, 10), (1100003, 17), (1100003, 16)])
def test_crowded_everywhere(n, S):
    follow(n, S, lattice(n, 1.2 * S))


@pytest.mark.parametrize("path", ["sparse", "dense"])
@pytest.mark.parametrize("n, S, spot, spacing", [(6000, 20, 3000, 0.2), (20000, 40, 8000, 0.25),
                                                 (20000, 40, 8000, 0.09), (140003, 60, 64000, 0.3),
                                                 (1100000, 110, 100000, 0.2),
                                                 (1100000, 110, 30000, 0.09)])
def test_dense_spots(n, S, spot, spacing, path):
    m = int(np.ceil(spot ** (1 / 3) - 1e-9))
    at = lattice(spot, m * spacing) + 1.2 * (S // 3) + 0.07
    rest = np.random.default_rng(n).uniform(0, 1.2 * S, (n - spot, 3))
    follow(n, S, np.concatenate([rest, at]), path=path)


@pytest.mark.parametrize("n, S, steps", [(5000, 165, 2), (140000, 165, 2), (1100000, 200, 2),
                                         (3000, 330, 1)])
def test_nearly_empty(n, S, steps):
    follow(n, S, np.random.default_rng(S).uniform(0, 1.2 * S, (n, 3)), steps)


def test_ensemble_with_a_crowded_replica():
    """A replica of 4^3 cells with 150 particles each beside dilute ones: the
    trajectories are those of the replicas by themselves."""
    sizes = [(9600, 4), (500, 20), (3000, 16)]
    integ = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=0.01, seed=5)
    pos = [lattice(n, 1.2 * S) for n, S in sizes]
    geom = [ps.SystemGeometry(n=n, box=1.2 * S, cells_per_dim=S, cell_size=1.2, integer=False)
            for n, S in sizes]
    with ps.Ensemble([ps.Replica(g, FREE) for g in geom], integ) as e:
        e.set_state(np.concatenate(pos))
        e.step(5)
        e.sync()
        together = e.get_state()["pos"]
    first = 0
    for g, p in zip(geom, pos):
        with ps.GpuSystem(g, FREE, integ, kernel_path="sparse") as s:
            s.set_state(p)
            assert s.step(5) in (0, ps.ERR_OVERLAP)
            alone = s.get_state()["pos"]
        if first == 0:   # the noise is keyed by the concatenated index
            assert np.array_equal(together[:g.n], alone)
        first += g.n
    assert np.isfinite(together).all()


def test_records_of_a_crowded_box():
    """The states that the rebuild records for the adjoint, 62 particles per cell
    (split): gradients with every state recorded are those of the recomputed
    segments."""
    n, S, K = 4000, 4, 6
    g = ps.SystemGeometry(n=n, box=28.0, cells_per_dim=S, cell_size=7.0, integer=False)
    mods = ps.AOPotential(kT=1.0, well_depth=0.3, cutoff=1.1)
    integ = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, seed=5)
    w = np.random.default_rng(8).standard_normal((n, 3))
    out = []
    with ps.GpuSystem(g, mods, integ) as s:
        s.set_state(ps.rsa_positions(n, g.box, 2))
        with ps.Adjoint(s, K, 3) as adj:
            for on in (False, True):
                adj.set_record_all(on)
                assert adj.forward() == 0
                out.append(adj.backward(w, with_gx0=True))
    assert np.abs(out[0]["gx0"]).max() > 0
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k
