"""The largest grid a context takes, 1290^3 cells, with a few particles (needs a
GPU with 40 GB free): pairs inside and across the box's faces against the
Calibration force written out, and three steps."""
import numpy as np
import pytest

import proteinsim2015_amd as ps

pytestmark = pytest.mark.gpu


def test_largest_grid():
    S, n = 1290, 64
    L = 1.2 * S
    g = ps.SystemGeometry(n=n, box=L, cells_per_dim=S, cell_size=1.2, integer=False)
    rng = np.random.default_rng(1)
    a = rng.uniform(0, L, (n // 2, 3))
    k = np.arange(12)
    a[k, k % 3] = (k % 2) * L + rng.uniform(-0.3, 0.3, 12)   # across the faces
    d = rng.normal(size=(n // 2, 3))
    d *= rng.uniform(0.95, 1.1, (n // 2, 1)) / np.linalg.norm(d, axis=1, keepdims=True)
    pos = np.mod(np.concatenate([a, a + d]), L)
    dd = pos[n // 2:] - pos[:n // 2]
    dd -= L * np.round(dd / L)
    r2 = (dd * dd).sum(1, keepdims=True)
    f = -36.0 * r2 ** -19.0 * dd
    integ = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, seed=1)
    with ps.GpuSystem(g, ps.Calibration(cutoff=1.15), integ) as s:
        s.set_state(pos)
        st, got = s.forces_now()
        assert st == 0 and s.step(3) == 0
        out = s.get_state()
    want = np.concatenate([f, -f])
    # r^-38: 38 times the relative error of a distance of two coordinates near L
    assert np.abs(got - want).max() <= 38 * 4 * np.spacing(L) * np.abs(want).max()
    moved = out["pos"] - pos
    moved -= L * np.round(moved / L)
    assert np.isfinite(out["pos"]).all() and 0 < np.abs(moved).max() < 0.1
