"""Positions outside the box or not finite in the thread-per-particle gather
(needs a GPU).  A particle that is nowhere (NaN, infinite) is no one's
neighbour: the strict r^2 < cutOff^2 (LJPotential.cpp:82) is false for it.  A
particle beyond the box is met in the image that the 27-cell walk meets it in,
as the brick kernel does, whose forces are the same bits.  The expected values
are those of the same particles without the strays, and of the brick kernel."""
import ctypes as C

import numpy as np
import pytest

import proteinsim2015_amd as ps
from proteinsim2015_amd import _lib

pytestmark = pytest.mark.gpu

CAL = {"cutOff": 2.5, "kT": 1.0}
LJ = {"cutOff": 2.5, "kT": 1.0, "wellDepth": 1.0, "yukawaStrength": 0.0, "ljNum": 6,
      "debyeLength": 0.5}
AO = {"cutOff": 1.1, "kT": 1.0, "wellDepth": 0.3}
MODULES = {"Cal": CAL, "LJ": LJ, "AO": AO}
INTEG = ps.BrownianIntegrator(kT=1.0, gamma=1.0, dt=1e-4, seed=1)


def geometry(n, S, cell):
    return ps.SystemGeometry(n=n, box=S * cell, cells_per_dim=S, cell_size=cell, integer=False)


def modules(name):
    return ps.PLUGINS[name].from_config(ps.Config(MODULES[name]))


def system(name, n, S, path):
    return ps.GpuSystem(geometry(n, S, 2.5), modules(name), INTEG, kernel_path=path)


def noalloc(sysg, pos):
    """psim_gpu_forces_noalloc with the system's parameters."""
    import torch
    d_pos = torch.tensor(pos, dtype=torch.float64, device="cuda").contiguous()
    d_f = torch.empty_like(d_pos)
    st = _lib.load().psim_gpu_forces_noalloc(C.byref(sysg.params), C.c_void_p(d_pos.data_ptr()),
                                             C.c_void_p(d_f.data_ptr()), None)
    torch.cuda.synchronize()
    return st, d_f.cpu().numpy()


def table(pos, g):
    """The reference's arrays for pos: cells in order, particles by index."""
    with np.errstate(invalid="ignore"):
        q = np.floor(pos / g.cell_size)
        q = np.where(q >= 0, np.minimum(q, g.cells_per_dim - 1), 0).astype(np.int64)
    key = q[:, 0] + g.cells_per_dim * (q[:, 1] + g.cells_per_dim * q[:, 2])
    order = np.argsort(key, kind="stable")
    start = np.searchsorted(key[order], np.arange(g.ncell))
    end = np.searchsorted(key[order], np.arange(g.ncell), side="right")
    cse = np.where((end > start)[:, None], np.stack([start, end], 1), -1)
    return (np.c_[pos[order], np.full(len(pos), g.radius)],
            np.stack([key[order], order], 1).astype(np.int32), cse.astype(np.int32))


@pytest.mark.parametrize("name", ["Cal", "LJ", "AO"])
@pytest.mark.parametrize("n, S", [(200, 3), (700, 6)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_particles_that_are_nowhere(name, n, S, bad):
    """Strays with one, two and three bad coordinates among ordinary ones near
    every face: the others' forces and neighbour sets are those without them."""
    g = geometry(n, S, 2.5)
    pos = ps.rsa_positions(n, g.box, 5)
    stray = np.arange(0, n, 29)
    for k, i in enumerate(stray):
        pos[i, :k % 3 + 1] = bad
        pos[i, k % 3 + 1:] = (0.01, g.box - 0.01)[k % 2]
    rest = np.setdiff1d(np.arange(n), stray)
    with system(name, n, S, "sparse") as s, system(name, len(rest), S, "sparse") as r:
        s.set_state(pos)
        r.set_state(pos[rest])
        st, f = s.forces_now()
        str_, fr = r.forces_now()
        cnt, _ = s.pair_stats()
        cntr, _ = r.pair_stats()
        stt, ft = s.force_table(*table(pos, g))
        stn, fn = noalloc(s, pos)
        assert s.last_error()[0] == 0
    assert st == str_ == stt == stn == 0
    assert not f[stray].any() and not cnt[stray].any()
    assert np.array_equal(f[rest], fr) and np.array_equal(cnt[rest], cntr)
    assert np.array_equal(ft, f) and np.array_equal(fn, f)


def test_a_stray_does_not_spread_in_steps():
    """Ten steps beside a particle that is NaN from the start."""
    n, S = 700, 6
    g = geometry(n, S, 2.5)
    pos = ps.rsa_positions(n, g.box, 6)
    pos[17] = np.nan
    with system("LJ", n, S, "sparse") as s:
        s.set_state(pos)
        assert s.step(10) == 0
        out = s.get_state()
    assert np.isnan(out["pos"][17]).all()
    assert np.isfinite(np.delete(out["pos"], 17, 0)).all()
    assert np.isfinite(np.delete(out["frc"], 17, 0)).all()


@pytest.mark.parametrize("name", ["Cal", "LJ"])
@pytest.mark.parametrize("S", [3, 4, 6])
@pytest.mark.parametrize("boxes", [-1e9, -70000.0, -3.0, -1.0, -0.4, 0.4, 1.0, 1.6, 3.0, 70000.0, 1e9])
def test_particles_beyond_the_box(name, S, boxes):
    """A tenth of the particles moved by whole and broken boxes, some of them
    together: every force has the brick kernel's bits."""
    n = 30 * S * S
    g = geometry(n, S, 2.5)
    pos = ps.rsa_positions(n, g.box, 7)
    rng = np.random.default_rng(S)
    far = rng.permutation(n)[:n // 10]
    pos[far, rng.integers(0, 3, len(far))] += boxes * g.box
    pos[far[1::2]] = pos[far[::2]][:len(far[1::2])] + [1.1, 0.2, 0.1]
    out = []
    for path in ("sparse", "brick"):
        with system(name, n, S, path) as s:
            s.set_state(pos)
            st, f = s.forces_now()
            out.append((st, f, *s.pair_stats()))
            if path == "sparse":
                stt, ft = s.force_table(*table(pos, g))
    assert out[0][0] == out[1][0] == stt
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.array_equal(ft, out[0][1], equal_nan=True)


def test_beyond_the_box_one_lane_per_particle():
    """262,144 particles (one lane each) and an ensemble of two systems."""
    n = 262144
    g = ps.SystemGeometry.exact(n, 0.05, 2.5)
    pos = ps.rsa_positions(n, g.box, 8)
    pos[::101, 0] += g.box
    pos[::103, 1] -= 2 * g.box
    pos[::997] = np.nan
    pos[::1009, 2] = np.inf
    out = []
    for path in ("sparse", "brick"):
        with ps.GpuSystem(g, modules("LJ"), INTEG, kernel_path=path) as s:
            s.set_state(pos)
            st, f = s.forces_now()
            out.append((f, *s.pair_stats()))
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)


def test_ensemble_with_strays():
    """Two replicas with strays: the pair statistics of the thread-per-particle
    kernel are those of each system by itself."""
    S, sizes = 6, (700, 333)
    g = [geometry(n, S, 2.5) for n in sizes]
    pos = [ps.rsa_positions(n, gg.box, 9 + n) for n, gg in zip(sizes, g)]
    for p in pos:
        p[5] = np.nan
        p[11, 0] += 2 * g[0].box
        p[40, 1] = -np.inf
    with ps.Ensemble([ps.Replica(gg, modules("LJ")) for gg in g], INTEG) as e:
        e.set_state(np.concatenate(pos))
        cnt, _ = e.pair_stats()
    want = []
    for gg, p in zip(g, pos):
        with ps.GpuSystem(gg, modules("LJ"), INTEG, kernel_path="brick") as s:
            s.set_state(p)
            want.append(s.pair_stats()[0])
    assert np.array_equal(cnt, np.concatenate(want))
