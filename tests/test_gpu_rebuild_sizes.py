"""A step's binning, sort and list build as one kernel against the three
kernels apart (the profile pass steps with those), the same states and
rebuilds bitwise, at the edges of what takes one kernel: just inside and
outside the largest number of workgroups, more particles than the binning
workgroups take in one pass, unequal particles with one type and with several.
Each case asserts which side it is on."""
import ctypes as C

import numpy as np
import pytest

from femmd_old_amd import System, configs

pytestmark = pytest.mark.gpu

REBUILD_MAX, BIN_PASS = 1024, 160 * 256


def _unequal(n, types):
    m = int(np.ceil(np.sqrt(n)))
    L = m * 1.2
    rng = np.random.default_rng(n)
    g = (np.arange(m) + 0.5) * (L / m)
    X, Y = np.meshgrid(g, g)
    s = System(L, L, dt=0.004)
    if types > 1:
        def table(lo, hi):
            a = rng.uniform(lo, hi, (types, types))
            return ((a + a.T) / 2).ravel()
        s.set_pair_potential(table(0.5, 1.5), table(1.6, 2.6), table(-0.05, 0.05))
    s.add_particles(X.ravel()[:n], Y.ravel()[:n], rng.normal(0, 0.9, n), rng.normal(0, 0.9, n),
                    rng.choice([1.0, 1.5], n), rng.uniform(0.9, 1.1, n),
                    rng.integers(0, types, n) if types > 1 else None)
    s.allocate_cuda()
    return s


def _one_rebuild(s):
    one, wgs = C.c_int32(), C.c_int32()
    assert s._lib.fm_test_one_rebuild(s.handle, C.byref(one), C.byref(wgs)) == 0
    return bool(one.value), wgs.value


@pytest.mark.parametrize("build,inside,lo,hi,passes", [
    (lambda: configs.build_system(configs.c2(scale=0.05)), True, 400, 700, 2),
    (lambda: configs.build_system(configs.c2(scale=0.1)), True, 970, 1000, 3),
    (lambda: configs.build_system(configs.c2(scale=0.105)), True, 1000, REBUILD_MAX, 3),
    (lambda: configs.build_system(configs.c2(scale=0.11)), False, REBUILD_MAX + 1, 1060, 4),
    (lambda: _unequal(5003, 1), True, 40, 200, 1),
    (lambda: _unequal(5003, 6), True, 40, 200, 1),
    (lambda: _unequal(45000, 6), True, 400, REBUILD_MAX, 2),
])
def test_one_kernel_rebuild_at_its_edges(build, inside, lo, hi, passes):
    a, b = build(), build()
    for s in (a, b):
        s.set_tuning(block=256)
        one, wgs = _one_rebuild(s)
        assert one == inside and lo <= wgs <= hi, (one, wgs)
        assert -(-s.N // BIN_PASS) == passes, s.N
    a.run(61)
    b.profile(60)  # advances 60 + 1 steps
    for u, v in zip(a.get_state(), b.get_state()):
        np.testing.assert_array_equal(u, v)
    assert a.list_stats() == b.list_stats()
    assert a.list_stats()["rebuilds"] > 2
    for s in (a, b):
        assert s.device_errors() == 0
        s.close()
