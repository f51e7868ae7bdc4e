"""Scenes whose rays walk their objects one after another, by the wave or each
lane for itself: closest hits, hit leaves and any-hits equal the
one-ray-per-lane kernel's for waves of neighbouring rays, of rays in all
directions and of both, part-filled waves, non-finite and zero directions,
small visit caps, 3 objects and more than 64 (which are never spread over a
wave's lanes)."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[3, 70])
def scene(gpu_ctx, request):
    objs, off = [], 0
    for k in range(request.param):
        soup = re.random_tris(k + 1, 2100 // request.param, -2.0, 2.0, 0.05, 0.4)
        objs.append(re.SceneObject(re.KDTree(soup), location=(0.3 * k % 2, 0.1 * k % 1.5, 0.0), rotation_y=0.4 * k,
                                   is_character=k == 2, prim_offset=off))
        off += len(soup)
    s = gpu_ctx.upload_scene(objs)
    s.n_obj = request.param
    yield s
    s.release()


def _rays(kind, n):
    rng = np.random.default_rng(n)
    o = rng.uniform(-5, 5, (n, 3))
    d = rng.uniform(-2, 2, (n, 3)) - o
    co, cd = re.camera_rays(re.Camera(pos=(0.3, 0.5, 6.0), view=(0.0, -0.1, -1.0)), 1024, n // 1024 + 1)
    i = np.arange(n)
    near = {"random": np.zeros(n, bool), "near": np.ones(n, bool), "waves": i // 64 % 2 == 0, "one": i % 64 != 17}[kind]
    o[near], d[near] = co[:n][near], cd[:n][near]
    o, d = o.astype(np.float32), d.astype(np.float32)
    for k, v in enumerate((0.0, np.nan, np.inf)):
        d[777 + 6400 * k] = v
    return o, d


# several objects are walked one after another above 393,216 walks (any-hit) and 1,179,648 (closest hit)
@pytest.mark.parametrize("kind", ["random", "near", "waves", "one"])
@pytest.mark.parametrize("cap", [1, 50])
def test_same_hits(scene, kind, cap):
    n = 1_200_031 // scene.n_obj + 20_000 if scene.n_obj <= 64 else 150_001
    o, d = _rays(kind, n)
    for one_sided in (True, False):
        kw = dict(one_sided=one_sided, max_leaf_visits=cap)
        want = scene.trace_closest(o, d, with_obj=True, variant=0, **kw)
        for block in (0, 256):
            got = scene.trace_closest(o, d, with_obj=True, variant=4, block=block, **kw)
            for a, b in zip(got, want):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), block
        any0 = scene.trace_closest(o, d, variant=0, secondary=True, **kw)[0] >= 0
        for block in (0, 128):
            assert np.array_equal(scene.occluded(o, d, block=block, **kw), any0.astype(np.uint8)), block
    c0, c4 = (scene.trace_counts(o, d, variant=v, **kw) for v in (0, 4))
    assert c0[2] == c4[2]
