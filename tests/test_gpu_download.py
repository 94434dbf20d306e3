"""Results through the pinned ring (csrc/download.hpp) against the same arrays
copied one at a time below its threshold: particle numbers at which arrays end
at a slot's end, one element before it and after it, with more slots' worth of
data than there are slots."""
import ctypes as C

import numpy as np
import pytest

from spatialpy_amd import _abi, workloads
from spatialpy_amd.engine import Engine

pytestmark = pytest.mark.gpu
SLOT = 2 << 20           # PinnedRing::SLOT
DOWNLOAD_MIN = 8 << 20

WIDTH = dict(x=3, v=3, vt=3, F=3, Fbp=3, rho=1, Frho=1, bvf_phi=1, nu=1, old_rho=1)


def read(eng, names):
    out = {k: np.zeros((eng.sa.n, WIDTH[k])) for k in names}
    st = _abi.State()
    for k, a in out.items():
        setattr(st, k, a.ctypes.data_as(C.POINTER(C.c_double)))
    assert eng.lib.ssasdpd_get_state(eng.h, C.byref(st)) == 0
    return out


# 8-byte elements of a slot: 262,144; particles of 24 bytes: 87,381, three times
# that is 262,143
@pytest.mark.parametrize("n", [SLOT // 8 - 1, SLOT // 8, SLOT // 8 + 1])
def test_state_through_the_ring(n):
    rng = np.random.default_rng(n)
    k = np.arange(n)
    x = np.stack([k % 64, k // 64 % 64, k // 4096], axis=1) * 0.1 + rng.uniform(-0.01, 0.01, (n, 3))
    sa = workloads.SystemArrays(
        x=x, type=np.ones(n, np.int32), mass=np.full(n, 1e-3), rho=np.ones(n), nu=np.full(n, 0.01), fixed=np.zeros(n, np.int32),
        n_types=1, dimension=3, h=0.13, dt=1e-5, nt=2, output_steps=np.array([0, 2], np.uint32), static_domain=0, rho0=1.0,
        c0=10.0, P0=100.0, bbox=workloads.bounding_box(x), v=rng.standard_normal((n, 3)), enable_rdme=False,
        enable_pde=False)
    eng = Engine(sa.normalized())
    eng.reset(seed=1)
    eng.advance(2)
    alone = {}
    for name in WIDTH:
        assert 8 * WIDTH[name] * n < DOWNLOAD_MIN
        alone.update(read(eng, [name]))
    assert np.isfinite(alone["F"]).all() and (alone["F"] != 0).any()
    for names in (list(WIDTH), ["x", "rho"], ["v", "F", "nu"]):    # [x, rho]: below, at and above the threshold
        for name, a in read(eng, names).items():
            assert np.array_equal(a, alone[name]), name


def test_counts_of_a_batch_through_the_ring():
    sa = workloads.static_rd_3d(n_side=20, nA=3000, nB=3000, t_end=0.2, num_points=3, dt=0.1)
    seeds = np.arange(40)
    eng = Engine(sa)
    many = eng.run_batch(seeds, fields=())["xx"]
    assert many.nbytes > DOWNLOAD_MIN
    for b in (0, 1, 17, 39):
        one = eng.run(seed=int(seeds[b]), fields=("xx",))["xx"]
        assert one.nbytes < DOWNLOAD_MIN
        assert np.array_equal(one, many[b])
