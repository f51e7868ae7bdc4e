"""The noise fill's two brick sizes and two gradient forms give the oracle's
bits: volumes on both sides of the size rule, cells aligned with the blocks
and not, negative origins, cells much smaller and much larger than a block."""
import numpy as np
import pytest

import oracle
import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (104, 104, 96), (104, 101, 104), (128, 128, 128)])
@pytest.mark.parametrize("kw", [
    dict(spacing=1 / 128), dict(spacing=(1 / 104, 1 / 101, 1 / 96)), dict(spacing=0.3, lacunarity=1.7, octaves=7),
    dict(spacing=1 / 1024, origin=(-3.3, 0.5, -0.01)), dict(spacing=1 / 128, octaves=0), dict(spacing=1 / 128, gain=-0.7),
])
def test_fill_equals_oracle(gpu_ctx, dims, kw):
    kw = dict(kw, spacing=tuple(np.broadcast_to(kw["spacing"], 3).astype(float)))
    vol = gpu_ctx.noise_volume(dim=dims, seed=11, **kw)
    got = vol.read()
    vol.release()
    want = oracle.noise_fill(re.perlin_table(11), dim=dims, **kw)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_coordinates_beyond_the_fast_forms(gpu_ctx):
    # the third octave's frequency overflows to infinity: the general kernel, NaN wherever the oracle has it
    kw = dict(dim=(20, 12, 9), spacing=(0.1,) * 3, octaves=3, lacunarity=1e30)
    vol = gpu_ctx.noise_volume(**kw)
    got = vol.read()
    vol.release()
    want = oracle.noise_fill(re.perlin_table(2016), **kw)
    assert np.array_equal(got, want, equal_nan=True)
