"""Every 64-point chunk of a training batch counts once: batches of one chunk,
around one and two chunks per block (256 blocks on a whole device), odd and
even, with the loss concentrated in one chunk, against the FP64 oracle (the
gradient bars of the surrogate's other tests: cosine 0.995, relative L2 0.1;
the loss of targets far from the outputs to 1 %)."""
import numpy as np
import pytest

import oracle
import rayengine_amd as re

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [1, 2, 3, 255, 256, 257, 511, 512, 513])
@pytest.mark.parametrize("where", ["first", "last"])
def test_loss_in_one_chunk(gpu_ctx, chunks, where):
    net = re.Surrogate(gpu_ctx, seed=3)
    params = net.params()[0]
    rng = np.random.default_rng(chunks)
    n = 64 * chunks
    s = np.concatenate([rng.random((n, 3)), rng.uniform(-0.1, 0.1, (n, 1))], 1).astype(np.float32)
    at = 0 if where == "first" else n - 64
    s[at:at + 64, 3] = 50.0
    loss, grad = net.batch_step(s, over_weight=4.0)
    net.release()
    # every other chunk's contribution is far below 1 % of this one's
    want_loss, want = oracle.mlp_loss_grad(params, s[:, :3], s[:, 3], 4.0)
    assert abs(loss - want_loss) <= 0.01 * want_loss
    cos = float(grad @ want) / (np.linalg.norm(grad) * np.linalg.norm(want))
    assert cos >= 0.995 and np.linalg.norm(grad - want) <= 0.1 * np.linalg.norm(want)
