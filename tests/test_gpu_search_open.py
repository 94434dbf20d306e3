"""The fixed-radius search where points have coordinates that are not finite:
they are nobody's neighbours, and the lists of the others stay exact however far
apart these are (the dimension has one cell then)."""
import ctypes as C

import numpy as np
import pytest

from spatialpy_amd import _abi
from spatialpy_amd.core.errors import SimulationError
from spatialpy_amd.engine import fr_search

pytestmark = pytest.mark.gpu


def pairs_and(extra, m):
    """m pairs at a distance of 0.5, 1e4 from one another along y, and points
    with the given y."""
    k = np.arange(m)
    p = np.zeros((2 * m, 3))
    p[0::2, 0] = p[1::2, 0] = (k % 7) * 0.9
    p[0::2, 1], p[1::2, 1] = k * 1e4, k * 1e4 + 0.5
    p[:, 2] = np.arange(2 * m) * 1e-4
    return np.concatenate([p, np.array([[0.3, y, 0.1] for y in extra]).reshape(-1, 3)])


# 300 and 4,000: a tree of one workgroup, and one with levels above
@pytest.mark.parametrize("m", [300, 4000])
@pytest.mark.parametrize("extra", [(), (np.nan,), (np.inf,), (-np.inf,), (np.inf, np.nan), (np.inf, -np.inf),
                                   (-np.inf, np.inf, np.inf)])
def test_lists_beside_a_point_that_is_not_finite(extra, m):
    p = pairs_and(extra, m)
    rows, idx, r2 = fr_search(p, p[:2 * m], 3, 0.6)
    assert np.array_equal(rows, np.arange(2 * m + 1))
    assert np.array_equal(idx, np.arange(2 * m) ^ 1)
    d = p[:2 * m] - p[idx]
    assert np.array_equal(r2, (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2])


@pytest.mark.parametrize("m", [300, 4000])
def test_x_from_minus_to_plus_infinity_is_refused(m):
    """No cut of dimension 0 separates such points: both calls of the protocol
    say so, the one for the lengths alone too."""
    p = pairs_and((), m)
    p[0, 0], p[1, 0] = -np.inf, np.inf
    with pytest.raises(SimulationError):
        fr_search(p, p[2:], 3, 0.6)
    lib, rows = _abi.load_library(), np.zeros(2 * m - 1, np.int64)
    q, ptr = np.ascontiguousarray(p[2:]), lambda a, t: a.ctypes.data_as(C.POINTER(t))
    assert lib.ssasdpd_fr_search(ptr(p, C.c_double), 2 * m, ptr(q, C.c_double), 2 * m - 2, 3, 0.6,
                                 ptr(rows, C.c_int64), None, None) != 0
