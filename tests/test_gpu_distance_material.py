"""The distance volume of an edited volume has a material channel of its own:
both keep their values when the other is edited or released, in either order,
and no release fails."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


def _edited(ctx):
    vol = ctx.noise_volume(dim=(24, 24, 24), spacing=(1 / 24,) * 3, seed=3)
    vol.edit("sphere_add", center=(0.5, 0.4, 0.5), extent=(0.2, 0.2, 0.2), material=3.0)
    return vol


@pytest.mark.parametrize("first", ["distance", "field"])
def test_either_volume_may_go_first(gpu_ctx, first):
    vol = _edited(gpu_ctx)
    mat = vol.read_material()
    assert (mat == 3.0).any()
    dist = re.distance_volume(vol)
    assert np.array_equal(dist.read_material(), mat)
    if first == "distance":
        dist.release()
        kept = vol
    else:
        vol.release()
        kept = dist
    # volumes that would take the place of one freed too early
    others = [_edited(gpu_ctx) for _ in range(4)]
    assert np.array_equal(kept.read_material(), mat)
    kept.edit("sphere_subtract", center=(0.5, 0.4, 0.5), extent=(0.3, 0.3, 0.3), material=7.0)
    assert (kept.read_material() == 7.0).any()
    for v in others:
        assert np.array_equal(v.read_material(), mat)
        v.release()
    kept.release()
    # an error left by a release would fail the next launch's check
    plain = gpu_ctx.noise_volume(dim=(8, 8, 8), spacing=(1 / 8,) * 3)
    re.distance_volume(plain).release()
    plain.release()
