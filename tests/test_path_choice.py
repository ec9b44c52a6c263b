"""Which pair kernel a context steps with (CPU only): choose_path compiled for
the host, on both sides of each of its lines.  The GPU tests of the wave-per-
cell kernel rely on these: kernel_info names both cell kernels "dense"."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or shutil.which("hipcc", path="/opt/rocm/bin")

PROGRAM = r"""
#include <cstdio>
#include "psim_params.hpp"
#include "psim_step.hpp"
int main() {
    int n, S, path;
    while (std::scanf("%d %d %d", &n, &S, &path) == 3) {
        psim_params P{};
        P.n_particles = n;
        P.cells_per_dim = S;
        P.box = 2.5 * S;
        P.cell_size = P.cutoff = 2.5;
        P.kernel_path = path;
        psim::Geo g;
        psim::Pot p;
        psim::GB b;
        psim::make_constants(P, g, p, b);
        const psim::PathChoice c = psim::choose_path(P, g);
        std::printf("%s\n", c.brick ? "brick" : !c.dense ? "particle" : c.cells ? "wave" : "workgroup");
    }
}
"""

AUTO, SPARSE, DENSE, BRICK = 0, 1, 2, 3
CASES = [
    # two particles per cell, and S = 3
    (1999, 10, AUTO, "particle"), (2000, 10, AUTO, "workgroup"), (5000, 3, AUTO, "particle"),
    (5000, 3, DENSE, "particle"),
    # 12,288 particles and 3.5 per cell
    (12287, 18, AUTO, "workgroup"), (12288, 18, AUTO, "wave"),
    (27999, 20, AUTO, "wave"), (28000, 20, AUTO, "workgroup"),
    (12301, 30, AUTO, "particle"), (12301, 30, DENSE, "wave"), (12301, 30, SPARSE, "particle"),
    (30011, 21, BRICK, "brick"),
    # the systems of test_gpu_cells.py and test_gpu_cells_stats.py
    (13000, 16, DENSE, "wave"), (13000, 17, DENSE, "wave"), (30011, 21, AUTO, "wave"),
    (15552, 18, AUTO, "wave"), (int(2.2 * 18 ** 3), 18, DENSE, "wave"),
    (int(5.5 * 18 ** 3), 18, DENSE, "workgroup"),
]


@pytest.mark.skipif(HIPCC is None, reason="hipcc not available")
def test_lines(tmp_path):
    src, exe = tmp_path / "choice.hip", tmp_path / "choice"
    src.write_text(PROGRAM)
    subprocess.check_call([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I",
                           os.path.join(ROOT, "include"), "-I",
                           os.path.join(ROOT, "proteinsim2015_amd", "csrc"), str(src), "-o",
                           str(exe)])
    out = subprocess.check_output([str(exe)], text=True,
                                  input="\n".join(f"{n} {S} {p}" for n, S, p, _ in CASES))
    for case, got in zip(CASES, out.split()):
        assert got == case[3], case
    assert len(out.split()) == len(CASES)
