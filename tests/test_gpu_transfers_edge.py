"""The state's round trip (test_gpu_transfers.py) on both sides of a full staging
buffer (needs a GPU): the five arrays, each padded to 64 bytes, take 8 MiB up to
69,904 particles and go through in one round, from 69,905 on in chunks."""
import pytest

from test_gpu_transfers import test_state_round_trip as round_trip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [69904, 69905])
def test_both_sides_of_a_full_buffer(n):
    padded = (24 * n + 63) // 64 * 64
    assert (5 * padded <= 8 << 20) == (n == 69904)
    round_trip(n)
