"""The device's reciprocal by one Newton step stands in for the IEEE quotient
also outside its range: rays whose directions have zero, tiny, huge and
infinite components, and triangles whose determinant is far beyond it, give
the oracle's hits and distances bit for bit."""
import numpy as np
import pytest

import oracle
import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1, 3, 4, 5])
@pytest.mark.parametrize("scale", [1.0, 1e-6, 1e6, 1e15])
def test_extreme_rays_and_triangles(gpu_ctx, variant, scale):
    rng = np.random.default_rng(5)
    tri = (re.random_tris(3, 300, -2.0, 2.0, 0.5, 3.0) * np.float32(scale)).astype(np.float32)
    tree = re.KDTree(tri)
    n = 1000
    o = (rng.uniform(-3, 3, (n, 3)) * scale).astype(np.float32)
    d = rng.standard_normal((n, 3)).astype(np.float32)
    d[::7, 0] = 0.0
    d[1::7, 1] = -0.0
    d[2::7, 2] = 1e-39
    d[3::7, 0] = 1e-38
    d[4::7] *= np.float32(1e18)
    d[5::49, 0] = np.inf
    scene = gpu_ctx.upload_scene([re.SceneObject(tree)])
    p, t = scene.trace_closest(o, d, variant=variant)
    scene.release()
    po, to = oracle.trace(*tree.export(), tree.identity_object(), o, d)
    assert np.array_equal(p, po) and np.array_equal(t.view(np.uint32), to.view(np.uint32))
