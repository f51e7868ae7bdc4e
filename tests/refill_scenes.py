"""Launches that variant 5 refills its waves in: more than 786,432 rays on one
object of more than 100,000 triangle records (others are launched as variant
4, so with three objects)."""
import numpy as np

import rayengine_amd as re

N_RAYS = 800_003


def refill_scene(ctx, n_obj):
    objs, off = [], 0
    for k in range(n_obj):
        soup = re.random_tris(k + 1, 30000 // n_obj, -2.0, 2.0, 0.05, 0.5)
        objs.append(re.SceneObject(re.KDTree(soup), location=(0.7 * k, 0.1 * k, 0.0), rotation_y=0.4 * k,
                                   is_character=k == 2, prim_offset=off))
        off += len(soup)
    scene = ctx.upload_scene(objs)
    assert len(scene.export()[2]) > 100_000
    return scene


def refill_rays(n=N_RAYS):
    rng = np.random.default_rng(n)
    o = rng.uniform(-5, 5, (n, 3))
    d = rng.uniform(-2, 2, (n, 3)) - o
    return o.astype(np.float32), d.astype(np.float32)
