"""Scenes of many objects: the exported scene is the concatenation of the
trees' records whether an object's records are copied by themselves or
gathered with its neighbours' (sizes on both sides of the 256 KiB an array is
gathered below, single, in runs and mixed), the objects' own records answer
rays, and an upload does not pay for every small object what one upload
costs."""
import time

import numpy as np
import pytest

import oracle
import rayengine_amd as re
from test_gpu_scene_place import _concatenated

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def trees():
    # 4,096 leaf records of 64 bytes or 6,554 triangle records of 40 are 256 KiB
    return {n: re.KDTree(re.random_tris(n, n, -2.0, 2.0, 0.1, 0.3), max_leaf_tris=4) for n in (1, 12, 700, 9000)}


@pytest.mark.parametrize("sizes", [(12,), (9000,), (12,) * 40, (9000, 12, 12, 9000, 12), (12, 9000, 9000, 1, 700),
                                   (700,) * 9, tuple([1, 12, 700] * 100)])
@pytest.mark.parametrize("offsets", [False, True])
def test_export_is_the_concatenation(gpu_ctx, trees, sizes, offsets):
    objs, off = [], 0
    for k, n in enumerate(sizes):
        objs.append(re.SceneObject(trees[n], location=(0.3 * k, 0.0, 0.0), prim_offset=off))
        off += n if offsets else 0
    scene = gpu_ctx.upload_scene(objs)
    for got, want, what in zip(scene.export(), _concatenated(objs), ("nodes", "leaves", "tris")):
        assert got.tobytes() == want.tobytes(), what
    rng = np.random.default_rng(len(sizes))
    o = rng.uniform(-3.0, 3.0, (500, 3)).astype(np.float32)
    d = rng.standard_normal((500, 3)).astype(np.float32)
    got = scene.trace_closest(o, d)
    want = oracle.trace(*scene.export(), o, d)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32))
    scene.release()


def test_small_objects_cost_less_than_uploads(gpu_ctx, trees):
    def best(n):
        objs = [re.SceneObject(trees[12], location=(k, 0.0, 0.0)) for k in range(n)]
        ts = []
        for _ in range(7):
            t = time.perf_counter()
            scene = gpu_ctx.upload_scene(objs)
            ts.append(time.perf_counter() - t)
            scene.release()
        return min(ts)

    # about 450 uploads of one object with copies and a launch for each
    assert best(1000) < 100 * best(1)
