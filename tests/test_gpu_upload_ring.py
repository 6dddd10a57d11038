"""GPU: host blocks gathered through the pinned ring (two slots of 98304 values; up to 196608
values in one slot), bit for bit as in test_gpu_upload.py: just below and above what one
slot takes, whole turns only, several turns with a remainder."""
import pytest

from test_gpu_upload import test_block_of_the_active_pairs as block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nO, nC, nR", [(32, 8, 0, 0), (32, 9, 0, 0), (32, 24, 0, 0), (48, 4, 0, 12), (60, 6, 0, 0),
                                           (61, 20, 1, 2)])
def test_turns_of_the_ring(n, nO, nC, nR):
    block(n, nO, nC, nR)
