"""The cooperative leaf test's list: lists of one entry to many windows of 512,
leaves of one triangle to hundreds, empty leaves among them; hits of the
one-ray-per-lane kernel, bit for bit."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf,depth", [(1, 30), (8, 30), (9, 3), (40, 6), (64, 5), (600, 2), (3000, 1)])
@pytest.mark.parametrize("one_sided", [True, False])
def test_list_windows(gpu_ctx, leaf, depth, one_sided):
    rng = np.random.default_rng(leaf)
    soup = re.random_tris(leaf, 2500, -2.0, 2.0, 0.05, 0.6)
    scene = gpu_ctx.upload_scene([re.SceneObject(re.KDTree(soup, max_leaf_tris=leaf, max_depth=depth))])
    for n in (5, 64, 700):
        o = rng.uniform(-5, 5, (n, 3)).astype(np.float32)
        d = (rng.uniform(-2, 2, (n, 3)) - o).astype(np.float32)
        for oo, dd in ((o, d), (np.repeat(o[:1], n, 0), np.repeat(d[:1], n, 0))):   # apart, and all in one leaf
            p0, t0 = scene.trace_closest(oo, dd, variant=0, one_sided=one_sided)
            for variant in (4, 5):
                p, t = scene.trace_closest(oo, dd, variant=variant, one_sided=one_sided)
                assert np.array_equal(p, p0) and np.array_equal(t, t0), (n, variant)
            assert np.array_equal(scene.occluded(oo, dd, one_sided=one_sided, secondary=False), (p0 >= 0).astype(np.uint8))
    scene.release()
