"""Straddlers clipped to their cells on the device: long slivers, triangles far
larger than the cells and faces along the cell planes give the host's tree,
byte for byte."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


def _soup(kind, n):
    rng = np.random.default_rng(n)
    if kind == "large":
        v = rng.uniform(-3, 3, (n, 3, 3))
    elif kind == "slivers":
        a = rng.uniform(-3, 3, (n, 1, 3))
        v = a + np.concatenate([np.zeros((n, 1, 3)), rng.uniform(-5, 5, (n, 1, 3)), rng.uniform(-1e-3, 1e-3, (n, 1, 3))], 1)
    else:                                  # corners on a lattice: vertices and edges on the planes
        v = rng.integers(-4, 5, (n, 3, 3)) / 4.0
    return v.reshape(n, 9).astype(np.float32)


@pytest.mark.parametrize("kind", ["large", "slivers", "lattice"])
@pytest.mark.parametrize("n,leaf,depth", [(1, 1, 8), (33, 1, 10), (200, 2, 12), (700, 4, 9)])
def test_clipped_trees(gpu_ctx, kind, n, leaf, depth):
    soup = _soup(kind, n)
    host = re.KDTree(soup, max_leaf_tris=leaf, max_depth=depth).export()
    dev = re.KDTree(soup, max_leaf_tris=leaf, max_depth=depth, ctx=gpu_ctx).export()
    for a, b in zip(host, dev):
        assert np.ascontiguousarray(a).tobytes() == np.ascontiguousarray(b).tobytes()
