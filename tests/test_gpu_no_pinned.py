"""An engine for which no pinned memory can be had gives what one with it
gives, bitwise: states below and above a transfer slot (1 MiB), forces,
energies and averages, a Hessian product, a gradient, the clusters'
observables, a batch's states, and the device's errors."""
import numpy as np
import pytest

from femmd_old_amd import Batch, FemmdError, System, configs

pytestmark = pytest.mark.gpu


def _pair(build):
    """The same system with and without."""
    out = [build(), build()]
    assert out[1]._lib.fm_test_pinned(out[1].handle, 0) == 0
    return out


def _same(a, b):
    if isinstance(a, dict):
        assert a.keys() == b.keys()
        for k in a:
            _same(a[k], b[k])
    elif isinstance(a, (list, tuple)):
        assert len(a) == len(b)
        for u, v in zip(a, b):
            _same(u, v)
    else:
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("scale", [0.01, 0.1])  # (the second: 23 k particles, 0.37 MiB)
def test_one_system(scale):
    a, b = _pair(lambda: configs.build_system(configs.c5(scale=scale, seed=3), commit=False))
    got = []
    for s in (a, b):
        s.allocate_cuda()
        s.run(25)
        x = s.get_state()
        s.set_state(x[0] + 1e-3, None, x[2], x[3])
        d = np.random.default_rng(1).normal(0, 1, (2, s.N))
        ids = np.arange(s.N)[::7].astype(np.int32)
        t = np.stack([x[0][ids], x[1][ids]], 1)
        got.append(dict(x=x, f=s.get_forces(), e=s.energies(), av=s.averages(), j=s.force_jvp(*d),
                        c=s.cluster_props(unfolded=True), w=s.cluster_virial(),
                        g=s.adjoint(12, ids, t, ckpt=5), end=s.get_state(), err=s.device_errors()))
    _same(*got)
    assert np.abs(got[0]["f"][0]).max() > 0 and got[0]["err"] == 0
    for s in (a, b):
        s.close()


def test_state_of_many_slots():
    n = 3 * (1 << 18) // 4 + 5  # four arrays: more than three slots
    rng = np.random.default_rng(2)
    m = int(np.ceil(np.sqrt(n)))
    cell = rng.permutation(m * m)[:n]
    x, y = (cell % m + 0.5) * 1.3, (cell // m + 0.5) * 1.3
    v = rng.normal(size=(2, n)).astype(np.float32)

    def build():
        s = System(1.3 * m, 1.3 * m, dt=0.001)
        s.add_particles(x, y, v[0], v[1])
        return s

    a, b = _pair(build)
    got = []
    for s in (a, b):
        s.allocate_cuda()
        s.run(3)
        s.set_state(y, x, v[1], v[0])
        s.run(2)
        got.append((s.get_state(), s.get_forces()))
    _same(*got)
    for s in (a, b):
        s.close()


def test_batch_and_device_error():
    ws = configs.c4(n_replicas=3, n_min=300, n_max=900)
    got = []
    for on in (1, 0):
        systems = [configs.build_system(w, commit=False) for w in ws]
        for s in systems:
            assert s._lib.fm_test_pinned(s.handle, on) == 0
        b = Batch(systems)
        b.run(20)
        got.append([(b.get_state(r), b.energies(r)) for r in range(len(b))])
        b.close()
    _same(*got)
    # coincident particles (an infinite force) are reported and cleared either way
    def two():
        s = System(20.0, 20.0)
        s.add_particles([5.0, 5.0, 12.0], [5.0, 5.0, 12.0])
        return s

    for s in _pair(two):
        s.allocate_cuda()
        with pytest.raises(FemmdError, match="non-finite"):
            s.run(2)
        assert s.device_errors() & 8
        s.clear_errors()
        assert s.device_errors() == 0
        s.close()
