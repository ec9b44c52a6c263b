"""The integrator with four lanes per particle (thread-per-particle path of
small systems) against the one-lane integrator of the brick path, bit for bit,
at the sizes where lane groups can go wrong (needs a GPU): systems below one
wave, partial waves; first step, velocity steps, the crossing tracker, in-kernel
and injected noise."""
import numpy as np
import pytest

import proteinsim2015_amd as ps

pytestmark = pytest.mark.gpu

AO = ps.AOPotential(kT=1.0, well_depth=ps.AOPotential.well_depth_for_contact(4.0, 0.1),
                    cutoff=1.1)
LJ = ps.LennardJones(kT=1.0, well_depth=1.0, yukawa_strength=0.0, lj_num=6, cutoff=1.1,
                     debye_length=0.5)
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-3, vel_freq=1, seed=21)


@pytest.mark.parametrize("force", [AO, LJ], ids=["ao", "lj"])
@pytest.mark.parametrize("injected", [False, True])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 1001])
def test_same_bits_as_one_lane(n, injected, force):
    geom = ps.SystemGeometry(n=n, box=13.2, cells_per_dim=12, cell_size=1.1, integer=False)
    pos = ps.rsa_positions(n, geom.box, n)
    rng = np.random.default_rng(n)
    vel = 8.0 * rng.standard_normal((n, 3))   # some cross a face on the first step
    noise = rng.standard_normal((5, 6, n)) if injected else None
    out = []
    for path in ("sparse", "brick"):
        with ps.GpuSystem(geom, [force], INTEG, kernel_path=path) as s:
            s.set_state(pos, vel=vel)
            s.track_start()
            assert s.step(5, noise) == 0
            out.append([*(s.get_state()[k] for k in ("pos", "pos0", "vel", "frc", "memx")),
                        *s.get_tracker()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
