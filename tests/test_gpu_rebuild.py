"""A step's binning, sort and list build as one kernel against the three
kernels apart (the profile pass steps with those): the same states and the
same rebuilds, bitwise, for one workgroup of each, with elements, with
particle types, just inside and outside the largest size that takes one
kernel, and after a change of the tiles."""
import numpy as np
import pytest

from femmd_old_amd import System, configs

pytestmark = pytest.mark.gpu


def _liquid(n):
    m = int(np.ceil(np.sqrt(n)))
    L = m * 1.12
    rng = np.random.default_rng(n)
    g = (np.arange(m) + 0.5) * (L / m)
    X, Y = np.meshgrid(g, g)
    v = rng.normal(0, 1.0, (2, n)).astype(np.float32)
    s = System(L, L, dt=0.005)
    s.add_particles(X.ravel()[:n], Y.ravel()[:n], v[0], v[1])
    s.allocate_cuda()
    return s


SYSTEMS = {
    "100": lambda: _liquid(100),
    "c1": lambda: configs.build_system(configs.c1(seed=5)),
    "c2": lambda: configs.build_system(configs.c2(scale=0.02)),
    "c5": lambda: configs.build_system(configs.c5(scale=0.05)),
    "100k": lambda: _liquid(100_000),
    "190k": lambda: _liquid(190_000),
}


@pytest.mark.parametrize("which", list(SYSTEMS))
def test_one_kernel_rebuild_equals_three(which):
    a, b = SYSTEMS[which](), SYSTEMS[which]()
    for s in (a, b):
        s.set_tuning(block=256)
    for tile in (None, 8):
        if tile:
            for s in (a, b):
                s.set_tuning(tile_cells=tile)
        a.run(61)
        b.profile(60)  # advances 60 + 1 steps
        for u, v in zip(a.get_state(), b.get_state()):
            np.testing.assert_array_equal(u, v)
        assert a.list_stats() == b.list_stats()
    assert a.list_stats()["rebuilds"] > 4
    for s in (a, b):
        assert s.device_errors() == 0
        s.close()
