"""The list build's hit masks at the edges of their words: a lane's candidate
run in a staged row (three cells) just below and above 32 and 64 candidates,
with and without an exclusion group in the wavefront, tiles of whole and
partial workgroups.  The interacting sets equal the oracle's FP32 predicate
exactly, from fresh and from stale lists."""
import numpy as np
import pytest

import oracle as O
from femmd_old_amd import System, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("disk", [False, True])
@pytest.mark.parametrize("run", [9.0, 31.0, 33.0, 63.0, 65.0])
def test_runs_around_a_mask_word(run, disk, block):
    rho = 0.8
    side = np.sqrt(run / 3.0 / rho)  # cells of run / 3 particles
    skin = float(side - configs.RC_WCA - 0.01)
    nc = 9
    L = float(np.float32(nc * side * 1.0005))
    rng = np.random.default_rng(int(run))
    m = int(L * np.sqrt(rho))
    g = (np.arange(m) + 0.5) * (L / m)
    X, Y = np.meshgrid(g, g)
    x, y = X.ravel(), Y.ravel()
    radius = 3.0
    if disk:
        keep = np.hypot(x - L / 2, y - L / 2) > radius + 1.0
        x, y = x[keep], y[keep]
    x = (x + rng.uniform(-0.05, 0.05, x.size)).astype(np.float32)
    y = (y + rng.uniform(-0.05, 0.05, y.size)).astype(np.float32)
    s = System(L, L, dt=0.004)
    s.set_skin(skin)
    s.add_particles(x, y, rng.normal(0, 0.7, x.size), rng.normal(0, 0.7, x.size))
    excl = -np.ones(x.size, np.int32)
    if disk:
        v, t = configs.hex_disk(radius, 1.0)
        s.add_elastomer(v.ravel(), t.ravel(), L / 2, L / 2, index_base=0, node_mass=1.0, E=50.0)
        excl = np.concatenate([excl, np.zeros(v.shape[0], np.int32)])
    s.allocate_cuda()
    s.set_tuning(block=block)
    ncx, ncy, _, _, _ = s.cells()
    assert ncx == nc and ncy == nc
    Lf = O.box_f32(L)
    for step in range(3):
        xc, yc, _, _ = s.get_state()
        cnt, s1, s2 = s.pair_sets()
        ocnt, os1, os2 = O.pair_sets(O.OracleSystem(Lf, Lf, xc, yc, excl=excl,
                                                    rc=np.array([np.float32(2 ** (1 / 6))])), 1)
        np.testing.assert_array_equal(cnt, ocnt)
        np.testing.assert_array_equal(s1, os1)
        np.testing.assert_array_equal(s2, os2)
        s.run(3)
    assert s.device_errors() == 0
    s.close()
