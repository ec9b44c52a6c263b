"""Shape of the cell rebuild's bins and tiles (CPU only): shape_bins compiled for
the host, over particle numbers, cells per dimension and cell volumes; the test
checks what the rebuild kernels rely on."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or shutil.which("hipcc", path="/opt/rocm/bin")

PROGRAM = r"""
#include <cstdio>
#include "psim_bins.hpp"
int main() {
    long long ncell;
    int n;
    double volume;
    while (std::scanf("%d %lld %lf", &n, &ncell, &volume) == 3) {
        psim::BinStore t;
        psim::shape_bins(n, (int)ncell, volume, t);
        std::printf("%d %d %d %d %d %d %d %d %d\n", t.lanes, t.per, (int)t.split, t.b.cap, t.b.cell_step,
                    t.b.member_step, t.b.shift, t.tiles, t.b.chains);
    }
}
"""

SIZES = [1, 7, 1000, 4096, 10000, 30011, 131071, 131072, 300007, 1048575, 1048576, 2097152, 60000000]
GRIDS = [3, 4, 5, 8, 13, 20, 31, 60, 100, 165, 330, 600, 1290]
LINE = [(3600, 4, 0), (3800, 4, 1), (10000, 4, 1), (30011, 4, 1), (24800, 6, 1), (140000, 11, 0),
        (140000, 10, 1), (1100003, 17, 0), (1100003, 16, 1)]
VOLUMES = [0.01, 1.33, 15.6, 27.0, 3e4]


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    if HIPCC is None:
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("bins")
    src, exe = d / "bins.hip", d / "bins"
    src.write_text(PROGRAM)
    subprocess.check_call([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I",
                           os.path.join(ROOT, "include"), "-I",
                           os.path.join(ROOT, "proteinsim2015_amd", "csrc"), str(src), "-o",
                           str(exe)])
    cases = [(n, S ** 3, v) for n in SIZES for S in GRIDS for v in VOLUMES]
    cases += [(n, S ** 3, 1.73) for n, S, _ in LINE]
    out = subprocess.check_output([str(exe)], text=True,
                                  input="\n".join(f"{n} {c} {v}" for n, c, v in cases))
    rows = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(rows) == len(cases)
    return list(zip(cases, rows))


def test_tiles_cover_the_cells(shapes):
    for (n, ncell, _), (lanes, per, split, cap, cell_step, member_step, shift, tiles, chains) in shapes:
        assert per in (4, 8) and 4 <= 1 << shift <= per * 256
        assert (tiles - 1) << shift < ncell <= tiles << shift


def test_a_mean_tile_is_moved_at_once(shapes):
    """A workgroup moves 256 particles per lane's share at once; where a tile of
    four cells holds more, the rebuild is split."""
    for (n, ncell, v), (lanes, per, split, cap, cell_step, member_step, shift, tiles, chains) in shapes:
        mean = n / ncell * (1 << shift)
        assert split or mean <= 256 * lanes, (n, ncell, v)
        assert not split or n / ncell > 50


def test_bins_are_addressed_apart(shapes):
    for (n, ncell, v), (lanes, per, split, cap, cell_step, member_step, shift, tiles, chains) in shapes:
        assert cap & (cap - 1) == 0
        if split:   # k_place reads whole rows, 16 members at a time
            assert (cell_step, member_step) == (cap, 1) and cap % 16 == 0
        else:
            assert (cell_step, member_step) == (1, ncell)


def test_memory_of_dilute_boxes(shapes):
    """Bins and chain heads stay within 256 bytes per particle or 1 GiB, or come
    down to 12 bytes per cell (8 bytes per cell is what the tables of counts and
    starts take by themselves)."""
    least = 0
    for (n, ncell, v), (lanes, per, split, cap, cell_step, member_step, shift, tiles, chains) in shapes:
        assert cap >= 1 and chains in (1, 4)
        assert cap == 1 or 4 * cap * ncell <= max(256 * n, 1 << 30), (n, ncell, v)
        if cap == 1 and ncell > 1 << 28:
            assert chains == 1
            least += 1
        if n / ncell > 1:   # the mean fits with room to spare
            assert cap > n / ncell or cap >= n
    assert least


def test_line_of_the_split_rebuild(shapes):
    """The systems of test_gpu_rebuild_crowded.py lie on the sides it names."""
    got = {c[:2]: r[2] for c, r in shapes}
    for n, S, split in LINE:
        assert got[n, S ** 3] == split, (n, S)
