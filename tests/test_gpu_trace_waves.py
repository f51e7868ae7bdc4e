"""Cooperative traversal with 8 to 64 rays a wave, the any-hit walk and the
refilled waves: the one-ray-per-lane kernel's hits, bit for bit, on both sides
of each launch-size limit."""
import numpy as np
import pytest
import torch

import rayengine_amd as re

pytestmark = pytest.mark.gpu


def _scene(ctx, n_obj, tris):
    objs, off = [], 0
    for k in range(n_obj):
        soup = re.random_tris(k + 1, tris // n_obj, -2.0, 2.0, 0.05, 0.5)
        objs.append(re.SceneObject(re.KDTree(soup), location=(0.7 * k, 0.1 * k, 0.0), rotation_y=0.4 * k,
                                   is_character=k == 2, prim_offset=off))
        off += len(soup)
    return ctx.upload_scene(objs)


def _rays(n):
    rng = np.random.default_rng(n)
    o = rng.uniform(-5, 5, (n, 3))
    d = rng.uniform(-2, 2, (n, 3)) - o
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("n_obj", [1, 3])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 65, 36864, 36865, 73728, 73729, 147456, 147457])
def test_rays_per_wave(gpu_ctx, n, n_obj):
    scene = _scene(gpu_ctx, n_obj, 3000)
    o, d = _rays(n)
    for one_sided in (True, False):
        p0, t0, k0 = scene.trace_closest(o, d, with_obj=True, variant=0, one_sided=one_sided)
        for variant, block in ((4, 0), (5, 0), (4, 128), (4, 256)):
            p, t, k = scene.trace_closest(o, d, with_obj=True, variant=variant, block=block, one_sided=one_sided)
            assert np.array_equal(p, p0) and np.array_equal(t, t0) and np.array_equal(k, k0), (variant, block)
        s0, _ = scene.trace_closest(o, d, variant=0, secondary=True, one_sided=one_sided)
        for block in (0, 128, 256):
            occ = scene.occluded(o, d, block=block, one_sided=one_sided)
            assert np.array_equal(occ, (s0 >= 0).astype(np.uint8)), block
    c0 = scene.trace_counts(o, d, variant=0)[2]
    assert scene.trace_counts(o, d, variant=5)[2] == c0
    scene.release()


@pytest.mark.parametrize("n_obj", [1, 3])
@pytest.mark.parametrize("n", [786432, 786433, 800000])
def test_refilled_waves(gpu_ctx, n, n_obj):
    scene = _scene(gpu_ctx, n_obj, 30000)  # more than 10^5 triangle records
    o, d = _rays(n)
    p0, t0, k0 = scene.trace_closest(o, d, with_obj=True, variant=0)
    p, t, k = scene.trace_closest(o, d, with_obj=True, variant=5)
    assert np.array_equal(p, p0) and np.array_equal(t, t0) and np.array_equal(k, k0)
    assert scene.trace_counts(o, d, variant=5)[2] == scene.trace_counts(o, d, variant=0)[2]
    do, dd = torch.as_tensor(o, device="cuda"), torch.as_tensor(d, device="cuda")
    hp, ht = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, device="cuda")
    hl = torch.empty(n, dtype=torch.int32, device="cuda")
    scene.trace_closest_hinted_device(do.data_ptr(), dd.data_ptr(), n, hp.data_ptr(), ht.data_ptr(),
                                      hit_leaf_ptr=hl.data_ptr(), variant=5)
    a = hl.cpu().numpy()
    assert np.array_equal(hp.cpu().numpy(), p0) and np.array_equal(ht.cpu().numpy(), t0)
    assert np.array_equal(a >= 0, p0 >= 0)
    scene.release()
