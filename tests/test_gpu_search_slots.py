"""The fixed-radius search around the list lengths past which it takes no
single-precision first pass: every point a neighbour of every other, on an engine
(whose hint is the last search's longest list) and in the stand-alone call."""
import numpy as np
import pytest

from spatialpy_amd import workloads
from spatialpy_amd.engine import Engine, fr_search

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [27, 28, 29, 30, 31, 32, 33, 34])
def test_lists_around_the_last_slots(n, oracle):
    x = np.random.default_rng(n).uniform(0, 0.01, (n, 3))
    for a, b in zip(fr_search(x, x, 3, 0.05), oracle.fr_search(x, x, 3, 0.05)):
        assert np.array_equal(a, b)
    sa = workloads.SystemArrays(
        x=x, type=np.ones(n, np.int32), mass=np.full(n, 1e-3), rho=np.ones(n), nu=np.full(n, 0.01),
        fixed=np.zeros(n, np.int32), n_types=1, dimension=3, h=0.05, dt=1e-9, nt=4, output_steps=np.array([0, 4], np.uint32),
        static_domain=0, bbox=workloads.bounding_box(x), enable_rdme=False, enable_pde=False)
    eng = Engine(sa.normalized())
    eng.reset(seed=1)
    eng.advance(4)
    rows, idx = eng.neighbors()[:2]
    # (the particle itself is in its list once it has moved)
    others = [set(idx[rows[i]:rows[i + 1]].tolist()) - {i} for i in range(n)]
    assert others == [set(range(n)) - {i} for i in range(n)]
