"""The refill kernel in every form a launch can ask for: visit caps, two-sided
and secondary rays, block sizes, counters, walk-start hints (the hit leaves of
the same rays, random ids in and out of range) with and without hit leaves,
the fixed scratch area, and the bounds-checked library; the one-ray-per-lane
kernel's hits, bit for bit.  The same for three objects, whose launches of
variant 5 are the plain cooperative kernel's."""
import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

import rayengine_amd as re
from rayengine_amd import _lib
from refill_scenes import N_RAYS, refill_rays, refill_scene

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def rays():
    o, d = refill_rays()
    return o, d, torch.as_tensor(o, device="cuda"), torch.as_tensor(d, device="cuda")


@pytest.fixture(scope="module", params=[1, 3])
def scene(gpu_ctx, request):
    s = refill_scene(gpu_ctx, request.param)
    yield s
    s.release()


def _same(a, b):
    return all(np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32)) for x, y in zip(a, b))


@pytest.mark.parametrize("one_sided", [True, False])
@pytest.mark.parametrize("secondary", [False, True])
@pytest.mark.parametrize("cap", [1, 3, 50, 4096])
def test_forms(scene, rays, cap, secondary, one_sided):
    o, d = rays[:2]
    kw = dict(max_leaf_visits=cap, secondary=secondary, one_sided=one_sided)
    want = scene.trace_closest(o, d, with_obj=True, variant=0, **kw)
    for block in (0, 128, 256):
        assert _same(scene.trace_closest(o, d, with_obj=True, variant=5, block=block, **kw), want), block
    c5, c0 = scene.trace_counts(o, d, variant=5, **kw), scene.trace_counts(o, d, variant=0, **kw)
    assert _same(c5[:2], want) and c5[2] == c0[2]


@pytest.mark.parametrize("block", [0, 128, 256])
@pytest.mark.parametrize("cap, one_sided", [(1, True), (50, True), (50, False), (4096, True)])
def test_hints(scene, rays, cap, one_sided, block):
    o, d, do, dd = rays
    kw = dict(max_leaf_visits=cap, one_sided=one_sided)
    want = scene.trace_closest(o, d, with_obj=True, variant=0, **kw)
    n_leaves = len(scene.export()[1])
    rng = np.random.default_rng(cap)
    # leaves of every object, ids past the last one and negative ones
    random_ids = rng.integers(-2, n_leaves + 50, N_RAYS).astype(np.int32)
    p = torch.empty(N_RAYS, dtype=torch.int32, device="cuda")
    t = torch.empty(N_RAYS, device="cuda")
    ob, hl = torch.empty_like(p), torch.empty_like(p)

    def run(start, leaves):
        for x in (p, ob, hl):
            x.fill_(-7)
        t.zero_()
        torch.cuda.synchronize()
        scene.trace_closest_hinted_device(do.data_ptr(), dd.data_ptr(), N_RAYS, p.data_ptr(), t.data_ptr(),
                                          start.data_ptr() if start is not None else 0,
                                          hl.data_ptr() if leaves else 0, ob.data_ptr(), variant=5, block=block, **kw)
        assert _same((p.cpu().numpy(), t.cpu().numpy(), ob.cpu().numpy()), want)
        return hl.cpu().numpy() if leaves else None

    first = run(None, True)
    assert np.array_equal(first >= 0, want[0] >= 0) and first.max() < n_leaves
    for start in (torch.as_tensor(first, device="cuda"), torch.as_tensor(random_ids, device="cuda")):
        run(start, False)
        assert np.array_equal(run(start, True) >= 0, want[0] >= 0)


def test_fixed_area(gpu_ctx, scene, rays):
    """Device pointers through the allocation-free call: two launches that take
    their rays from the area's counters, the second smaller, with counters."""
    o, d, do, dd = rays
    tp = re._trace_params(variant=5)
    for n in (N_RAYS, N_RAYS - 9000):
        p = torch.full((n,), -7, dtype=torch.int32, device="cuda")
        t = torch.zeros(n, device="cuda")
        torch.cuda.synchronize()
        cnt = (C.c_uint64 * 4)()
        st = _lib.lib().re_trace_closest_noalloc(gpu_ctx.handle, scene.id, do.data_ptr(), dd.data_ptr(), n,
                                                 C.byref(tp), p.data_ptr(), t.data_ptr(), None, cnt,
                                                 re.RE_DEVICE_PTRS)
        assert st == 0
        want = scene.trace_counts(o[:n], d[:n], variant=0)
        assert _same((p.cpu().numpy(), t.cpu().numpy()), want[:2]) and list(cnt) == list(want[2])


@pytest.mark.timeout(200, method="thread")
def test_bounds_checked_library():
    """tests/refill_bounds_child.py: a process holds one of the two libraries."""
    env = dict(os.environ, RE_LIBRARY="debug")
    print("refill bounds child: start", flush=True)
    r = subprocess.run([sys.executable, "-u", str(ROOT / "tests" / "refill_bounds_child.py")], env=env,
                       capture_output=True, text=True, timeout=180)
    print(r.stdout[-4000:], r.stderr[-4000:], flush=True)
    assert r.returncode == 0 and r.stdout.rstrip().endswith("refill bounds ok")
