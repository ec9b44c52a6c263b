"""Every pair kernel a context can step with has its neighbour statistics as a
kernel of its own (CPU only; the built library's kernels by name)."""
import pytest

from proteinsim2015_amd import _lib
from test_code_object import READELF, gfx950_code_objects, kernel_metadata


@pytest.mark.skipif(READELF is None, reason="llvm-readelf not available")
@pytest.mark.parametrize("step, stats", [("6k_step", "7k_stats"), ("12k_step_dense", "13k_stats_dense"),
                                         ("12k_step_cells", "13k_stats_cells"),
                                         ("12k_step_brick", "13k_stats_brick")])
def test_statistics_of_each_step_kernel(step, stats):
    names = {k for co in gfx950_code_objects(_lib.LIB_PATH) for k in kernel_metadata(co)}
    assert any(step in k for k in names)
    assert any(stats in k for k in names)
