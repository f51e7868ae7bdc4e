"""Work items cut to 8, 16, 32, 64 or more rays by the batch's ray count: the
single-workload results, ray for ray, on both sides of each limit, and the
plan's item count."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("total,item_rays", [(1, 256), (64, 7), (36864, 256), (36865, 256), (73729, 256), (147457, 256),
                                             (147457, 1), (6291455, 256), (6291456, 256), (12582912, 256),
                                             (12582912, 100)])
def test_cut_items(gpu_ctx, total, item_rays):
    rng = np.random.default_rng(total + item_rays)
    tree = re.KDTree(re.random_tris(1, 500, -2.0, 2.0, 0.2, 1.0))
    vol = gpu_ctx.noise_volume(dim=(24, 24, 24), spacing=(1 / 24,) * 3, seed=3)
    base = 4096                       # distinct rays, repeated
    o = rng.uniform(-3, 3, (base, 3)).astype(np.float32)
    d = (rng.uniform(0, 1, (base, 3)) - o).astype(np.float32)
    idx = np.arange(total) % base
    cut = total * 2 // 3
    b = re.Batch(gpu_ctx, [(tree, 0, cut)], [(vol, 0, cut, total - cut)], o[idx], d[idx], item_rays=item_rays)
    assert b.items() == -(-cut // item_rays) + -(-(total - cut) // item_rays)
    scene = gpu_ctx.upload_scene([re.SceneObject(tree)])
    p0, t0 = scene.trace_closest(o, d, variant=0)
    tm, hm, _, _ = re.hybrid_trace(vol, None, o, d)
    pm = np.where(hm == 1, 0, -1).astype(np.int32)
    want_p = np.where(np.arange(total) < cut, p0[idx], pm[idx])
    want_t = np.where(np.arange(total) < cut, t0[idx], tm[idx])
    for _ in range(2):
        b.run()
        p, t = b.results()
        assert np.array_equal(p, want_p) and np.array_equal(t, want_t)
        assert (b.completion_ms()[1:] > 0).all()
    b.release()
    scene.release()
    vol.release()
