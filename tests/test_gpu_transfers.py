"""State copies through the pinned staging buffer at the sizes where they can
go wrong (needs a GPU): below one page, both sides of one full buffer (8 MiB
of five arrays: 69,905 particles), many chunks with a remainder.  The export
of a state read right after a step (previous positions, forces and memory
still in the last step's slot order) must equal, bit for bit, the export after
they were gathered, and reading must not disturb the trajectory."""
import numpy as np
import pytest

import proteinsim2015_amd as ps

pytestmark = pytest.mark.gpu

LJ = {"cutOff": 2.5, "kT": 1.0, "wellDepth": 1.0, "yukawaStrength": 0.0, "ljNum": 6,
      "debyeLength": 0.5}


@pytest.mark.parametrize("n", [1, 170, 171, 69905, 69906, 200001])
def test_state_round_trip(n):
    geom = ps.SystemGeometry.exact(n, 0.05, 2.5) if n > 1000 else \
        ps.SystemGeometry(n=n, box=26.0, cells_per_dim=10, cell_size=2.6, integer=False)
    mods = ps.PLUGINS["LJ"].from_config(ps.Config(LJ))
    integ = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, vel_freq=2, seed=5)
    rng = np.random.default_rng(n)
    pos = ps.rsa_positions(n, geom.box, 3)
    vel = rng.normal(size=(n, 3))
    with ps.GpuSystem(geom, mods, integ) as a, ps.GpuSystem(geom, mods, integ) as b:
        a.set_state(pos, vel=vel)
        got = a.get_state()
        assert np.array_equal(got["pos"], pos) and np.array_equal(got["vel"], vel)
        b.set_state(pos, vel=vel)
        assert a.step(3) == 0 and b.step(3) == 0
        lagged = a.get_state()
        a.observables()              # gathers the arrays into the slot order
        settled = a.get_state()
        for k in lagged:
            assert np.array_equal(lagged[k], settled[k]), k
        a.step(2), b.step(1)
        b.get_state()                # a read between two steps
        b.step(1)
        ga, gb = a.get_state(), b.get_state()
        for k in ga:
            assert np.array_equal(ga[k], gb[k]), k
