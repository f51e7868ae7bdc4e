"""A call that finds the device full fails alone: the calls after it, launches
and builds, succeed."""
import numpy as np
import pytest

import oracle
import rayengine_amd as re
from rayengine_amd import _lib

pytestmark = pytest.mark.gpu


def test_calls_after_a_failed_allocation(small):
    import torch
    tri_v, tree, o, d = small
    ctx = re.Context(0)
    scene = ctx.upload_scene([re.SceneObject(tree)])
    # a host-pointer trace whose staging is twice the card: refused before any ray is read
    n = 2 * torch.cuda.mem_get_info()[1] // 36
    buf = np.zeros(16, np.float32)

    def full():
        st = _lib.lib().re_trace_closest(ctx.handle, scene.id, _lib.ptr(buf), _lib.ptr(buf), n, None, _lib.ptr(buf),
                                         _lib.ptr(buf), None, 0)
        assert _lib.STATUS_NAMES[st] == "RE_ERR_OOM"

    full()
    got = scene.trace_closest(o, d)
    want = oracle.trace(*tree.export(), tree.identity_object(), o, d)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32))
    full()
    built = re.KDTree(tri_v, ctx=ctx)
    assert all(a.tobytes() == b.tobytes() for a, b in zip(built.export(), tree.export()))
    scene.release()
    ctx.close()
