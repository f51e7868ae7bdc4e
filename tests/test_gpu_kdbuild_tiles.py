"""Device kd build at the sizes where its kernels' tiles end: nodes around the
64 references of the exact split, reference arrays around the chunks of the
partition.  The tree must equal the host build's byte for byte."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


def _equal(tri, ctx, **kw):
    host, dev = re.KDTree(tri, **kw), re.KDTree(tri, ctx=ctx, **kw)
    for a, b, what in zip(host.export(), dev.export(), ("nodes", "leaves", "tris")):
        assert a.tobytes() == b.tobytes(), f"{what} differ: n={len(tri)} {kw}"


@pytest.mark.parametrize("n", [1, 2, 9, 63, 64, 65, 1023, 1024, 1025, 2049])
@pytest.mark.parametrize("leaf,clip", [(1, True), (8, True), (8, False)])
def test_tile_edges(gpu_ctx, n, leaf, clip):
    # large triangles: most references straddle the first planes
    _equal(re.random_tris(n, n, -2.0, 2.0, 0.5, 3.0), gpu_ctx, max_leaf_tris=leaf, max_depth=16, clip=clip)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 140000])
def test_root_box_and_refusal(gpu_ctx, n):
    # bounds over the last partial block and past the grid's first round (512 blocks of 256); zeros of both signs
    tri = re.random_tris(n, n, -2.0, 2.0, 0.1, 1.0)
    tri[:, 4] = np.where(np.arange(n) % 3 == 0, np.float32(-0.0), np.float32(0.0))
    tri[:, 1], tri[:, 7] = np.abs(tri[:, 1]), np.abs(tri[:, 7])
    host, dev = re.KDTree(tri, max_depth=4), re.KDTree(tri, max_depth=4, ctx=gpu_ctx)
    for k in ("root_min", "root_max"):
        assert host.info[k].tobytes() == dev.info[k].tobytes(), k
    for at, bad in ((0, np.nan), (n - 1, np.inf), (n // 2, -np.inf)):
        worse = tri.copy()
        worse[at, 5] = bad
        with pytest.raises(re.ReError):
            re.KDTree(worse, ctx=gpu_ctx)
