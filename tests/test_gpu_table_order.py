"""psim_gpu_force_table on tables whose cells are not stored in row order
(needs a GPU).  A row of cells is read from its first non-empty cell's start to
its last one's end, which for such a table may end before it starts: that row
then has no candidates, and the rest of the table must not notice.  Expected
values: the ordered table's bits where no neighbour cell moved, and a walk over
the rows in numpy (relative 1e-11: pair terms r^-37 of FP64 sums in another
order)."""
import numpy as np
import pytest

import proteinsim2015_amd as ps

pytestmark = pytest.mark.gpu

RC = 2.5
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, seed=1)


def table(pos, g, cell_order):
    """The reference's arrays with the cells stored in cell_order."""
    S = g.cells_per_dim
    q = np.minimum((pos / g.cell_size).astype(np.int64), S - 1)
    key = q[:, 0] + S * (q[:, 1] + S * q[:, 2])
    place = np.empty(g.ncell, np.int64)
    place[cell_order] = np.arange(g.ncell)
    order = np.argsort(place[key], kind="stable")
    count = np.bincount(key, minlength=g.ncell)
    end = np.empty(g.ncell, np.int64)
    end[cell_order] = np.cumsum(count[cell_order])
    cse = np.where((count > 0)[:, None], np.stack([end - count, end], 1), -1)
    return order, key, cse.astype(np.int32)


def walk(pos, g, order, key, cse, particles):
    """Calibration forces of the row walk on the given particles."""
    S, x = g.cells_per_dim, pos[order]
    slot = np.empty(len(pos), np.int64)
    slot[order] = np.arange(len(pos))
    out = np.zeros((len(particles), 3))
    for k, i in enumerate(particles):
        cx, cy, cz = key[i] % S, key[i] // S % S, key[i] // S ** 2
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                row = (cy + dy) % S * S + (cz + dz) % S * S * S
                for cells in ([c for c in (cx - 1, cx, cx + 1) if 0 <= c < S],
                              [c % S for c in (cx - 1, cx + 1) if not 0 <= c < S]):
                    r = [cse[row + c] for c in cells if cse[row + c, 0] >= 0]
                    if not r:
                        continue
                    j = np.arange(r[0][0], r[-1][1])   # empty where it ends before it starts
                    j = j[j != slot[i]]
                    d = x[j] - pos[i]
                    d -= g.box * np.round(d / g.box)
                    r2 = (d * d).sum(1)
                    d, r2 = d[r2 < RC * RC], r2[r2 < RC * RC]
                    out[k] += ((-36.0 * r2 ** -19.0)[:, None] * d).sum(0)
    return out


@pytest.mark.parametrize("n, S, sample", [(700, 6, 700), (5000, 12, 400), (262144, 40, 150)])
@pytest.mark.parametrize("order", ["reversed", "two cells swapped"])
def test_cells_out_of_order(n, S, sample, order):
    g = ps.SystemGeometry(n=n, box=RC * S, cells_per_dim=S, cell_size=RC, integer=False)
    pos = ps.rsa_positions(n, g.box, 3)
    cells = np.arange(g.ncell)
    mid = S // 2 * (1 + S + S * S)
    if order == "reversed":
        cells = cells[::-1].copy()
    else:
        cells[[mid, mid + 1]] = cells[[mid + 1, mid]]
    print(f"table n={n} S={S} {order}", flush=True)
    with ps.GpuSystem(g, ps.Calibration(cutoff=RC), INTEG) as s:
        out = []
        for c in (np.arange(g.ncell), cells):
            o, key, cse = table(pos, g, c)
            st, f = s.force_table(np.c_[pos[o], np.full(n, 0.5)],
                                  np.stack([key[o], o], 1).astype(np.int32), cse)
            assert st == 0
            out.append(f)
    some = np.random.default_rng(n).permutation(n)[:sample]
    if order != "reversed":
        far = np.abs(np.stack([key % S, key // S % S, key // S ** 2], 1) - S // 2).max(1) > 2
        assert far.any() and np.array_equal(out[0][far], out[1][far])
        some = np.concatenate([some, np.where(~far)[0][:200]])
    for f, c in zip(out, (np.arange(g.ncell), cells)):
        want = walk(pos, g, *table(pos, g, c), some)
        assert np.abs(f[some] - want).max() <= 1e-11 * np.abs(want).max()
