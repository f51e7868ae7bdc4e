"""The device memory a context keeps between kd builds is given back when an
allocation of that context finds the device full, and the next build gives the
tree of the first."""
import ctypes as C

import numpy as np
import pytest

import rayengine_amd as re
from rayengine_amd import _lib

pytestmark = pytest.mark.gpu


def test_chunk_is_given_back_when_the_device_is_full():
    import torch
    ctx = re.Context(0)
    tri_v = re.random_tris(3, 60000, -2.0, 2.0, 0.05, 0.1)
    scene = ctx.upload_scene([re.SceneObject(re.KDTree(re.random_tris(1, 10, -1.0, 1.0, 0.1, 0.3)))])
    first = re.KDTree(tri_v, ctx=ctx).export()
    held, total = torch.cuda.mem_get_info()
    # a host-pointer trace whose staging is twice the card: refused before any ray is read
    n = 2 * total // 36
    buf = np.zeros(16, np.float32)
    st = _lib.lib().re_trace_closest(ctx.handle, scene.id, _lib.ptr(buf), _lib.ptr(buf), n, None, _lib.ptr(buf),
                                     _lib.ptr(buf), None, 0)
    assert _lib.STATUS_NAMES[st] == "RE_ERR_OOM"
    free, _ = torch.cuda.mem_get_info()
    assert free - held >= 8 << 20
    for a, b in zip(first, re.KDTree(tri_v, ctx=ctx).export()):
        assert a.tobytes() == b.tobytes()
    scene.release()
    ctx.close()
