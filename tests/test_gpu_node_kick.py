"""The node kick of systems without pair forces where it has many workgroups
(from 1024 a workgroup reads its corner forces through LDS, in chunks of 2048)
against the direct reading of each replica alone, bitwise: partial last
workgroups, more corners than a chunk, free particles between."""
import numpy as np
import pytest

from femmd_old_amd import Batch, System

pytestmark = pytest.mark.gpu


def _sheet(nx, ny, bonds, seed):
    rng = np.random.default_rng(seed)
    X, Y = np.meshgrid(np.arange(nx, dtype=np.float32), np.arange(ny, dtype=np.float32), indexing="ij")
    a = (np.arange(nx - 1)[:, None] * ny + np.arange(ny - 1)).ravel()
    t = np.concatenate([np.stack([a, a + ny, a + 1], 1), np.stack([a + ny, a + ny + 1, a + 1], 1)])
    v = np.stack([X.ravel(), Y.ravel()], 1) + rng.uniform(-0.05, 0.05, (nx * ny, 2))
    s = System(nx + 30.0, ny + 30.0, dt=0.002)
    s.set_lj(False)
    s.set_youngs_modulus(40.0, 0.3)
    free = rng.uniform(0, 20, (2, 333))
    s.add_particles(free[0], free[1], *rng.normal(0, 1, (2, 333)))
    n0 = s.add_elastomer(v.ravel(), t.ravel(), 10.0, 10.0, index_base=0, node_mass=1.0)
    # stretched bonds along every edge, or every seventh
    e = np.unique(np.sort(np.concatenate([t[:, [0, 1]], t[:, [1, 2]], t[:, [2, 0]]]), axis=1), axis=0)
    e = e[:: 1 if bonds else 7]
    s.add_bonds(n0 + e[:, 0], n0 + e[:, 1], 25.0, 0.97 * np.hypot(*(v[e[:, 0]] - v[e[:, 1]]).T))
    return s


SHEETS = [(210, 211, True), (200, 223, False), (215, 204, True), (199, 221, True), (223, 200, False),
          (212, 213, True)]


def test_gather_through_lds_equals_direct():
    alone, many = [], []
    for k, (nx, ny, bonds) in enumerate(SHEETS):
        alone.append(_sheet(nx, ny, bonds, k))
        many.append(_sheet(nx, ny, bonds, k))
    spans = [-(-s.N // 256) for s in alone]
    assert sum(spans) >= 1024 > 2 * max(spans)
    b = Batch(many)
    b.run(25)
    for r, s in enumerate(alone):
        s.allocate_cuda()
        x0 = s.get_state()
        s.run(25)
        for u, v, w in zip(b.get_state(r), s.get_state(), x0):
            np.testing.assert_array_equal(u, v)
            assert np.abs(v - w)[333:].max() > 0  # (the nodes moved)
        assert s.device_errors() == 0
        s.close()
    assert b.device_errors() == 0
    b.close()
