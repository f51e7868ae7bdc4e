"""The hybrid march with a network that never sends a ray on (no distance
exceeds tau, no ray travels far enough to come back): every ray is evaluated
once where it enters and then marches the exact field, so its distance, hit
and samples are those of the march without a network, which runs in another
kernel, one ray a lane and none refilled."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def field(gpu_ctx):
    vol = gpu_ctx.noise_volume(dim=(40, 33, 47), spacing=(1 / 47,) * 3, seed=4)
    net = re.Surrogate(gpu_ctx, seed=2)
    yield vol, net
    net.release()
    vol.release()


@pytest.mark.parametrize("max_iters", [1, 7, 4096])
@pytest.mark.parametrize("n", [1, 15, 17, 8193, 196608, 196609, 393217, 700001])
def test_rays_march_as_without_a_network(field, n, max_iters):
    vol, net = field
    rng = np.random.default_rng(n)
    o = rng.uniform(-0.3, 1.2, (n, 3)).astype(np.float32)
    d = (rng.uniform(0.1, 0.6, (n, 3)) - o).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    kw = dict(margin_voxels=1.0, k_exact=0.1, n_bisect=4, max_iters=max_iters)
    t, hit, evals, samples = re.hybrid_trace(vol, net, o, d, tau_voxels=1e30, rejoin_voxels=1e30, **kw)
    t0, hit0, evals0, samples0 = re.hybrid_trace(vol, None, o, d, **kw)
    assert np.array_equal(t.view(np.uint32), t0.view(np.uint32)) and np.array_equal(hit, hit0)
    assert np.array_equal(samples, samples0) and np.array_equal(evals, (samples0 > 0).astype(np.int32))
    assert not evals0.any()
    if n > 1000 and max_iters > 100:  # marches of many lengths: lanes are refilled
        assert len(np.unique(samples0)) > 20
