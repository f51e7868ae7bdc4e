"""Child process of test_gpu_refill_forms.py (RE_LIBRARY=debug is set by the
parent): the bounds-checked library's refill kernel, and with three objects its
plain cooperative one, as they are, counted and hinted, against the one-ray-per-lane kernel, with no
bounds-check bit set."""
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
sys.path[:0] = [str(ROOT), str(ROOT / "tests")]

import numpy as np  # noqa: E402
import torch  # noqa: E402  (one HIP runtime: torch's, loaded first)

import rayengine_amd as re  # noqa: E402
from rayengine_amd import _lib  # noqa: E402
from refill_scenes import N_RAYS, refill_rays, refill_scene  # noqa: E402


def main():
    assert _lib.LIB_PATH.name == "librayengine_debug.so", _lib.LIB_PATH
    ctx = re.Context(0)
    o, d = refill_rays()
    do, dd = torch.as_tensor(o, device="cuda"), torch.as_tensor(d, device="cuda")
    for n_obj in (1, 3):
        scene = refill_scene(ctx, n_obj)
        p0, t0 = scene.trace_closest(o, d, variant=0)
        n_leaves = len(scene.export()[1])

        def check(p, t, what):
            print(f"{n_obj} objects, {what}", flush=True)
            assert np.array_equal(p, p0) and np.array_equal(t.view(np.uint32), t0.view(np.uint32)), what
            m = ctx.debug_bounds_errors()
            assert m == 0, f"{what}: bounds-check bits {m:#x}"

        check(*scene.trace_closest(o, d, variant=5), "refill")
        check(*scene.trace_counts(o, d, variant=5)[:2], "refill, counted")
        p = torch.empty(N_RAYS, dtype=torch.int32, device="cuda")
        t = torch.empty(N_RAYS, device="cuda")
        hl = torch.empty_like(p)
        start = torch.as_tensor(np.random.default_rng(2).integers(-2, n_leaves + 50, N_RAYS).astype(np.int32),
                                device="cuda")
        torch.cuda.synchronize()
        scene.trace_closest_hinted_device(do.data_ptr(), dd.data_ptr(), N_RAYS, p.data_ptr(), t.data_ptr(),
                                          start.data_ptr(), hl.data_ptr(), variant=5)
        check(p.cpu().numpy(), t.cpu().numpy(), "refill, hinted")
        scene.release()
    ctx.close()
    print("refill bounds ok", flush=True)


if __name__ == "__main__":
    main()
