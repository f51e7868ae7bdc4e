"""Objects placed in a scene by the device: the exported scene equals the
trees' own records with entry, leaf, triangle and prim indices offset, for
object sizes around a work-group's 256 records and one to four objects."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


def _concatenated(objs):
    nodes, leaves, tris = [], [], []
    nb = lb = tb = 0
    for ob in objs:
        n, l, t = (a.copy() for a in ob.tree.export())
        meta = n["meta"].astype(np.int64)
        low, kind = meta & 0x3FFFFFFF, meta >> 30
        n["meta"] = ((kind << 30) | (low + np.where(kind == 3, lb, nb))).astype(np.uint32)
        r = l["rope"].astype(np.int64)
        r = np.where(r == -1, -1, np.where(r < -1, r + lb, r + nb))
        l["rope"] = r.astype(np.int32)
        l["first"] += tb
        t["prim"] += ob.prim_offset
        nodes.append(n)
        leaves.append(l)
        tris.append(t)
        nb, lb, tb = nb + len(n), lb + len(l), tb + len(t)
    return np.concatenate(nodes), np.concatenate(leaves), np.concatenate(tris)


@pytest.mark.parametrize("sizes", [(1,), (257,), (1, 1), (255, 256, 257), (1500, 1, 40, 700)])
@pytest.mark.parametrize("offsets", [False, True])
def test_export_is_the_concatenation(gpu_ctx, sizes, offsets):
    objs, off = [], 0
    for i, n in enumerate(sizes):
        objs.append(re.SceneObject(re.KDTree(re.random_tris(i, n, -2.0, 2.0, 0.1, 1.0), max_leaf_tris=2),
                                   prim_offset=off))
        off += n if offsets else 0
    scene = gpu_ctx.upload_scene(objs)
    for got, want, what in zip(scene.export(), _concatenated(objs), ("nodes", "leaves", "tris")):
        assert got.tobytes() == want.tobytes(), what
    scene.release()
