"""The counting sort at the edges of its blocks: cell counts (ncx * ncy and a
closing cell) around one and several blocks of 64 and around the count from
which blocks of 256 are taken, with few particles per cell and with more than
a block's LDS copy holds.  Within a cell the order is the caller's."""
import numpy as np
import pytest

from femmd_old_amd import System, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,skin", [(3, 0.6), (7, 0.6), (8, 0.6), (11, 0.6), (16, 0.6), (156, 0.6),
                                     (157, 0.6), (313, 0.6),
                                     (314, 0.6), (8, 3.4), (25, 3.4)])
def test_sorted_order(nc, skin):
    L = float(np.float32((nc + 0.5) * (configs.RC_WCA + skin)))
    rng = np.random.default_rng(nc)
    m = int(L * np.sqrt(0.88))
    g = (np.arange(m) + 0.5) * (L / m)
    X, Y = np.meshgrid(g, g)
    p = rng.permutation(m * m)  # caller order unrelated to the place
    x = (X.ravel()[p] + rng.uniform(-0.04, 0.04, p.size)).astype(np.float32)
    y = (Y.ravel()[p] + rng.uniform(-0.04, 0.04, p.size)).astype(np.float32)
    s = System(L, L, dt=0.002)
    s.set_skin(skin)
    s.add_particles(x, y, rng.normal(0, 0.7, p.size), rng.normal(0, 0.7, p.size))
    s.allocate_cuda()
    for _ in range(2):
        ncx, ncy, key, start, perm = s.cells()
        assert ncx == nc and ncy == nc
        np.testing.assert_array_equal(perm, np.lexsort((np.arange(p.size), key)))
        np.testing.assert_array_equal(start[1:], np.cumsum(np.bincount(key, minlength=nc * nc)))
        assert start[0] == 0
        s.run(12)
    assert s.device_errors() == 0
    s.close()
