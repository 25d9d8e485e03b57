"""Host arrays in and out of the engine at the edges of its transfer slots
(1 MiB, a ring of four): one value, a state just below, at and just above one
slot and past the ring, arrays that straddle two slots, a subset of the
arrays; before and after a re-ordering.  Values come back bitwise, positions
wrapped by the FP32 rule v - floor(v / L) L."""
import numpy as np
import pytest

from femmd_old_amd import System

pytestmark = pytest.mark.gpu

SLOT = (1 << 20) // 4  # floats


def _wrap(v, L):
    return v - np.floor(v / L) * L


@pytest.mark.parametrize("n", [1, 257, SLOT // 4 - 1, SLOT // 4, SLOT // 4 + 1, SLOT + 1])
def test_state_at_slot_edges(n):
    m = max(int(np.ceil(np.sqrt(n))), 8)
    L = np.float32(1.3 * m)
    rng = np.random.default_rng(n)
    cell = rng.permutation(m * m)[:n]  # caller order unrelated to the place
    x = ((cell % m + 0.5 + rng.uniform(-0.1, 0.1, n)) * 1.3).astype(np.float32)
    y = ((cell // m + 0.5 + rng.uniform(-0.1, 0.1, n)) * 1.3).astype(np.float32)
    v = rng.normal(size=(2, n)).astype(np.float32)
    s = System(float(L), float(L), dt=0.001)
    s.add_particles(x, y, v[0], v[1])
    s.allocate_cuda()
    for k in range(2):
        for a, b in zip(s.get_state(), (_wrap(x, L), _wrap(y, L), v[0], v[1])):
            np.testing.assert_array_equal(a, b)
        # one image up and down, then velocities alone
        up = (x + L * rng.integers(-1, 2, n).astype(np.float32)).astype(np.float32)
        x, y = y, up
        s.set_state(x, y, None, v[0])
        v[1] = v[0]
        for a, b in zip(s.get_state(), (_wrap(x, L), _wrap(y, L), v[0], v[1])):
            np.testing.assert_array_equal(a, b)
        v = rng.normal(size=(2, n)).astype(np.float32)
        s.set_state(None, None, v[0], v[1])
        f = s.get_forces()
        s.reorder()
        for a, b in zip(f, s.get_forces()):
            np.testing.assert_array_equal(a, b)
        x, y = _wrap(x, L), _wrap(y, L)
    assert np.abs(f[0]).max() < 1e3 and (n < 257 or np.abs(f[0]).max() > 0)
    assert s.device_errors() == 0
    s.close()
