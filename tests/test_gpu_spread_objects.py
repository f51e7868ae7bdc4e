"""A lane for every object of a ray: hits, objects, distances, hit leaves and
work counts of the walks one after another, on both sides of the limits."""
import numpy as np
import pytest
import torch

import rayengine_amd as re

pytestmark = pytest.mark.gpu


def _scene(ctx, n_obj):
    objs = []
    for k in range(n_obj):
        # some objects coincide: equal distances go to the first
        soup = re.random_tris(k // 2, 60, -1.0, 1.0, 0.1, 0.7)
        objs.append(re.SceneObject(re.KDTree(soup), location=(0.3 * (k // 2 % 5), 0.2 * (k // 2 % 3), 0.0),
                                   rotation_y=0.4 * (k // 2), is_character=k == 5, prim_offset=100 * k))
    return ctx.upload_scene(objs)


@pytest.mark.parametrize("n_obj", [2, 3, 7, 63, 64, 65])
@pytest.mark.parametrize("n", [1, 100, 6144, 18432, 18433, 60000])
def test_spread_equals_in_turn(gpu_ctx, n_obj, n):
    scene = _scene(gpu_ctx, n_obj)
    rng = np.random.default_rng(n)
    o = rng.uniform(-4, 4, (n, 3)).astype(np.float32)
    d = (rng.uniform(-1, 1, (n, 3)) - o).astype(np.float32)
    for one_sided in (True, False):
        ref = scene.trace_closest(o, d, with_obj=True, variant=0, one_sided=one_sided, secondary=True)
        for block in (0, 256):
            got = scene.trace_closest(o, d, with_obj=True, variant=4, block=block, one_sided=one_sided, secondary=True)
            assert all(np.array_equal(a, b) for a, b in zip(got, ref))
        occ = scene.occluded(o, d, one_sided=one_sided)
        assert np.array_equal(occ, (ref[0] >= 0).astype(np.uint8))
    assert scene.trace_counts(o, d, variant=4)[2] == scene.trace_counts(o, d, variant=0)[2]
    scene.release()


@pytest.mark.parametrize("n_obj", [2, 7])
def test_hinted_walks(gpu_ctx, n_obj):
    scene = _scene(gpu_ctx, n_obj)
    base, n = 500, 1200000 // n_obj              # the same rays in a small launch and beyond the limit
    rng = np.random.default_rng(1)
    o = rng.uniform(-4, 4, (base, 3)).astype(np.float32)
    d = (rng.uniform(-1, 1, (base, 3)) - o).astype(np.float32)
    out = []
    for m in (base, n):
        idx = np.arange(m) % base
        do, dd = torch.as_tensor(o[idx], device="cuda"), torch.as_tensor(d[idx], device="cuda")
        p, t = torch.empty(m, dtype=torch.int32, device="cuda"), torch.empty(m, device="cuda")
        ob, hl = torch.empty_like(p), torch.empty_like(p)
        start = torch.full_like(p, -1)
        for _ in range(2):                       # the second time from the first one's leaves
            cnt = scene.trace_closest_hinted_device(do.data_ptr(), dd.data_ptr(), m, p.data_ptr(), t.data_ptr(),
                                                    start_leaf_ptr=start.data_ptr(), hit_leaf_ptr=hl.data_ptr(),
                                                    obj_ptr=ob.data_ptr(), counts=True, variant=4)
            start = hl.clone()
            torch.cuda.synchronize()
        out.append([x[:base].cpu().numpy() for x in (p, t, ob, hl)])
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    ref = scene.trace_closest(o, d, with_obj=True, variant=0)
    assert all(np.array_equal(a, b) for a, b in zip((out[0][0], out[0][1], out[0][2]), ref))
    scene.release()
