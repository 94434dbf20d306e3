"""Neighbour lists in kd-tree visit order where the tree's build changes its
path: up to 1,024 points one workgroup splits everything, beyond that whole
levels run first and each cell of 1,024 points or fewer is finished alone.
Lattices are full of exact distance ties, which the visit order decides;
clusters make the tree deep and its cells uneven."""
import numpy as np
import pytest

from spatialpy_amd.engine import fr_search

pytestmark = pytest.mark.gpu


def points(kind, n, dim, rng):
    m = int(np.ceil(n ** (1.0 / dim)))
    x = np.zeros((n, 3))
    if kind == "lattice":
        g = np.meshgrid(*[np.arange(m)] * dim, indexing="ij")
        x[:, :dim] = np.stack([c.ravel() for c in g], axis=1)[rng.permutation(m ** dim)[:n]]
        return x, 1.5
    # half of the points in a corner a thousand times denser
    x[:, :dim] = rng.uniform(0, m, (n, dim))
    x[: n // 2, :dim] *= 1e-3
    return x, 0.05 if n > 100 else 1.0


@pytest.mark.parametrize("kind", ["lattice", "cluster"])
@pytest.mark.parametrize("n,dim", [(1, 3), (2, 3), (3, 1), (64, 2), (65, 3), (1023, 3), (1024, 2), (1025, 3),
                                   (2049, 1), (5000, 3), (9001, 2)])
def test_lists_follow_the_kdtree_at_every_size(kind, n, dim, oracle):
    x, h = points(kind, n, dim, np.random.default_rng(n))
    if kind == "cluster" and n > 1000:
        x[: n // 2, :dim] *= 100.0      # keep the lists short
    got, ref = fr_search(x, x, dim, h), oracle.fr_search(x, x, dim, h)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)
