"""The sky's form for a sun straight overhead: frames whose sun is overhead to
the bit take it, others the general form, and both stay within one 8-bit step
of the oracle on every pixel (the tolerance of the sky's hardware functions)."""
import numpy as np
import pytest

import oracle
import rayengine_amd as re
from rayengine_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sun", [(0.0, 1.0, 0.0), (-0.0, 1.0, -0.0), (0.0, 1.0, 1e-7), (0.0, 0.5, 0.0), (0.3, 0.8, 0.52)])
@pytest.mark.parametrize("width,height", [(64, 36), (33, 7)])
def test_sky_of_each_form(gpu_ctx, sun, width, height):
    _, d = re.camera_rays(W.TERRAIN_CAMERA, width, height)
    d[: len(d) // 2, 1] = np.abs(d[: len(d) // 2, 1])   # half of the view above the horizon
    hit = (np.arange(len(d)) % 5 == 0).astype(np.uint8)
    normal = np.tile(np.float32([0, 1, 0]), (len(d), 1))
    got = re.frame_shade(gpu_ctx, d, hit, normal, width, height, sun_dir=sun).view(np.uint8).astype(int)
    want = oracle.frame_shade(oracle.frame_params(sun_dir=sun), d, hit, normal, width, height).view(np.uint8).astype(int)
    assert np.abs(got - want).max() <= 1
