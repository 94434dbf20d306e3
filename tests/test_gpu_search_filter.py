"""The fixed-radius search tells most candidates apart in single precision and
compares the rest exactly: lists must be the oracle's, bit for bit, where that
could go wrong: distances at h to the last bit, positions far from the origin,
grids so wide that single precision resolves less than h, queries that are not
points, lists around the lengths at which the kernel changes."""
import numpy as np
import pytest

from spatialpy_amd.engine import fr_search

pytestmark = pytest.mark.gpu


def _case(kind, dim, rng):
    if kind == "at_h":              # lattice neighbours at 0.1, 0.2, ... and h among them
        g = np.meshgrid(*[np.arange(12) * 0.1] * dim, indexing="ij")
        x = np.stack([c.ravel() for c in g], axis=1)
        return x, x, 0.2
    if kind == "shifted":           # 1e6 h from the origin
        x = rng.uniform(0, 1, (1500, dim)) + 1e5
        return x, x, 0.1
    if kind == "wide":              # pairs a distance of h apart, to the last bits, along 3e6 h
        a = np.sort(rng.uniform(0, 3e5, 700))
        d = 0.1 * (1.0 + np.arange(-350, 350) * 2.0 ** -40)
        x = np.zeros((1400, dim))
        x[:, 0] = np.concatenate([a, a + d])
        return x, x, 0.1
    if kind == "queries":           # inside, beside and far outside the points
        x = rng.uniform(0, 1, (900, dim))
        q = np.concatenate([rng.uniform(-0.3, 1.3, (400, dim)), x[:50], np.full((3, dim), 1e12), np.full((2, dim), -50.0)])
        return x, q, 0.15
    n = int(kind)                   # everyone a neighbour of everyone: lists of n - 1
    x = rng.uniform(0, 0.01, (n, dim))
    return x, x, 0.05


@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("kind", ["at_h", "shifted", "wide", "queries", "2", "11", "12", "13", "16", "17", "24", "32",
                                  "33", "90"])
def test_lists_are_exact(kind, dim, oracle):
    x, q, h = _case(kind, dim, np.random.default_rng(dim))
    p3, q3 = np.zeros((len(x), 3)), np.zeros((len(q), 3))
    p3[:, :dim], q3[:, :dim] = x, q
    got, ref = fr_search(p3, q3, dim, h), oracle.fr_search(p3, q3, dim, h)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)
