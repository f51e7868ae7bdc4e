"""Training batches that take the blocks of the gradient kernel through its
loop two to four times, whole rounds and part-filled ones.

With over_weight 0 a point whose target lies below the output adds exactly
nothing, so the gradient of a batch is the sum of the gradients of the same
batch with one round's chunks left in at a time: the same BF16 operands and
products, only the FP32 additions in another order.  Those differ by about
1e-6 of a gradient's norm (rounding of sums of 10^5 terms of random sign), a
staged row of 128 points that is not what it should be by more than 1e-3 of
the norm of its weight block: the bar is 1e-4 for every block by itself, the
first layer's columns in two."""
import numpy as np
import pytest

import rayengine_amd as re

pytestmark = pytest.mark.gpu

# the flat parameters: W0 (features 0..63 and 64..98 apart), b0, W1, b1, ...
H, IN = 64, 99


def _blocks(grad):
    w0 = grad[:H * IN].reshape(H, IN)
    out = {"W0[:, :64]": w0[:, :64], "W0[:, 64:]": w0[:, 64:]}
    at = H * IN
    for name, n in [("b0", H), ("W1", H * H), ("b1", H), ("W2", H * H), ("b2", H), ("W3", H * H), ("b3", H),
                    ("W4", H), ("b4", 1)]:
        out[name] = grad[at:at + n]
        at += n
    assert at == grad.size
    return out


@pytest.mark.parametrize("rounds_of_blocks, extra", [(2, 1), (3, 0), (4, 0), (4, 1), (6, 1), (8, 0)])
def test_gradient_is_the_sum_of_its_rounds(gpu_ctx, rounds_of_blocks, extra):
    import torch
    blocks = torch.cuda.get_device_properties(0).multi_processor_count
    chunks = rounds_of_blocks * blocks + extra
    n = 64 * chunks
    rng = np.random.default_rng(chunks)
    s = np.empty((n, 4), np.float32)
    s[:, :3] = rng.random((n, 3))
    up = rng.uniform(20.0, 30.0, n).astype(np.float32)  # above every output: weight 1
    net = re.Surrogate(gpu_ctx, seed=11)

    def step(active):
        s[:, 3] = np.where(active, up, np.float32(-1e3))  # below: weight 0
        return net.batch_step(s, over_weight=0.0)

    loss, grad = step(np.ones(n, bool))
    again = step(np.ones(n, bool))
    round_of = np.arange(n) // 64 // (2 * blocks)
    parts = [step(round_of == r) for r in range(round_of[-1] + 1)]
    net.release()
    assert np.array_equal(grad.view(np.uint32), again[1].view(np.uint32)) and loss == again[0]
    assert len(parts) >= 2 and np.isfinite(grad).all()
    want = np.sum([p[1].astype(np.float64) for p in parts], axis=0)
    for (name, g), w in zip(_blocks(grad).items(), _blocks(want).values()):
        assert np.linalg.norm(g - w) <= 1e-4 * np.linalg.norm(w), name
    assert abs(loss - sum(p[0] for p in parts)) <= 1e-4 * loss
