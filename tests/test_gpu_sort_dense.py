"""The counting sort in blocks of 256 cells with more entries than one round
of its lanes takes (1024) and than its LDS copy holds (4096, the ranks then
read from memory), just above the cell count from which such blocks are
taken (24,576)."""
import pytest

from test_gpu_sort_blocks import test_sorted_order as check_sorted_order

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,skin,per_block", [(158, 1.9, (1200, 4096)), (158, 3.4, (4097, 5000))])
def test_sorted_order_of_dense_blocks(nc, skin, per_block):
    from femmd_old_amd import configs
    per_cell = 0.88 * (configs.RC_WCA + skin) ** 2
    assert nc * nc + 1 > 24576 and per_block[0] <= 256 * per_cell <= per_block[1]
    check_sorted_order(nc, skin)
