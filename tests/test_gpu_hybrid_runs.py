"""The hybrid march with 16, 32 and 64 rays a wave and refilled lanes: every
ray's distance, hit, evaluations and samples are those of the same ray in a
launch of its own size class, and of the exact march without the network."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def field(gpu_ctx):
    vol = gpu_ctx.noise_volume(dim=(40, 33, 47), spacing=(1 / 47,) * 3, seed=4)
    net = re.Surrogate(gpu_ctx, seed=2)
    dist = re.distance_volume(vol)
    net.train(dist, n_samples=1 << 14, batch=2048, steps=60, seed=3)
    dist.release()
    rng = np.random.default_rng(8)
    o = rng.uniform(-0.3, 1.2, (3000, 3)).astype(np.float32)
    d = (rng.uniform(0.1, 0.6, (3000, 3)) - o).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    yield vol, net, o, d
    net.release()
    vol.release()


@pytest.mark.parametrize("max_iters", [1, 7, 4096])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 8191, 8193, 196608, 196609, 393216, 393217, 700001])
def test_same_ray_same_result(field, n, max_iters):
    vol, net, o, d = field
    kw = dict(tau_voxels=4.0, margin_voxels=1.0, k_exact=0.1, n_bisect=4, max_iters=max_iters)
    # one ray per wave's worth of launches: a few rays alone, then repeated over the launch
    base = re.hybrid_trace(vol, net, o, d, **kw)
    idx = np.arange(n) * 7 % len(o)
    got = re.hybrid_trace(vol, net, o[idx], d[idx], **kw)
    for a, b in zip(got, base):
        assert np.array_equal(np.asarray(a).view(np.uint8 if a.dtype == np.uint8 else np.uint32),
                              np.asarray(b)[idx].view(np.uint8 if b.dtype == np.uint8 else np.uint32))
    assert (base[2] <= max_iters).all()
    one = [re.hybrid_trace(vol, net, o[k:k + 1], d[k:k + 1], **kw) for k in range(0, 12)]
    for j in range(4):
        assert np.array_equal(np.concatenate([x[j] for x in one]), base[j][:12])
