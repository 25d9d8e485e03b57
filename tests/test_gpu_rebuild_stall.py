"""A rebuild whose waits are given up (the bound set to no polls at all, so
every kernel ends at once): the run reports it, further runs of the handle give
up without waiting to their bound, and after clear_errors the handle steps as one
that never stalled, bitwise, through many more rebuilds."""
import time

import numpy as np
import pytest

from femmd_old_amd import FemmdError, System, configs

pytestmark = pytest.mark.gpu

STALL = 32  # FM_DEV_SORT_STALL


def _liquid(n):
    m = int(np.ceil(np.sqrt(n)))
    L = m * 1.12
    rng = np.random.default_rng(n)
    g = (np.arange(m) + 0.5) * (L / m)
    X, Y = np.meshgrid(g, g)
    v = rng.normal(0, 1.0, (2, n)).astype(np.float32)
    s = System(L, L, dt=0.002)
    s.add_particles(X.ravel()[:n], Y.ravel()[:n], v[0], v[1])
    return s


@pytest.mark.parametrize("build", [lambda: _liquid(900),
                                   lambda: configs.build_system(configs.c1(seed=5), commit=False)])
def test_a_stalled_rebuild_is_recovered(build):
    a, b = build(), build()
    lib = a._lib
    for s in (a, b):
        s.set_reorder_interval(0)
        s.allocate_cuda()
        s.set_tuning(block=256)
    start = a.get_state()
    assert lib.fm_test_rebuild_spins(a.handle, 0) == 0
    with pytest.raises(FemmdError, match="timed out"):
        for _ in range(60):
            a.run(5)
    assert a.device_errors() & STALL
    # more rebuilds before the error is cleared, at the usual bound (seconds):
    # each gives up long before it
    assert lib.fm_test_rebuild_spins(a.handle, -1) == 0
    t = time.perf_counter()
    with pytest.raises(FemmdError, match="timed out"):
        a.run(100)
    assert time.perf_counter() - t < 1.0
    a.clear_errors()
    assert a.device_errors() == 0
    # a stall in the first of a recorded trajectory's segments, whose next
    # ones bin and sort without the host between
    assert lib.fm_test_rebuild_spins(a.handle, 0) == 0
    a.set_state(*start)
    with pytest.raises(FemmdError, match="timed out"):
        a.adjoint_forward(160, 40)
    assert lib.fm_test_rebuild_spins(a.handle, -1) == 0
    a.clear_errors()
    a.set_state(*start)
    for s in (a, b):
        n0 = s.list_stats()["rebuilds"]
        s.run(200)
        assert s.list_stats()["rebuilds"] - n0 > 2
        assert s.device_errors() == 0
    for u, v in zip(a.get_state(), b.get_state()):
        np.testing.assert_array_equal(u, v)
    ea, eb = a.energies(), b.energies()
    assert all(ea[k] == eb[k] for k in ea if k != "steps")
    for s in (a, b):
        s.close()
