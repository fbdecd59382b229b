"""The warm-start network's tiled products at the sizes where they can go wrong: batches
and widths around the 64-wide padding, K below one step per wavefront, more layers than
one weight launch takes, both tile sizes; against the CPU oracle."""
import numpy as np
import pytest
import torch

import mlp_oracle as mo
from squander_hip import Context
from squander_hip.mlp import WarmStartMLP

pytestmark = pytest.mark.gpu


# (in, hidden, hidden layers, out, batch)
@pytest.mark.parametrize("shape", [(1, 1, 0, 1, 1), (64, 64, 1, 64, 64), (65, 63, 2, 129, 65), (130, 192, 10, 7, 33),
                                   (512, 1024, 1, 1000, 1000)])
def test_gradients_match_oracle(shape):
    """bf16 operands: 2e-2 of the oracle that rounds where the kernels do; the sums differ
    in order only, so most of that is the activations' own rounding."""
    ind, hid, nh, out, B = shape
    print(shape, flush=True)
    net = WarmStartMLP(Context(0), ind, hid, nh, out, seed=7)
    rng = np.random.default_rng(2)
    x = rng.standard_normal((B, ind)).astype(np.float32)
    t = rng.standard_normal((B, out)).astype(np.float32)
    loss, g = net.gradients(x, t)
    loss_o, g_o, _ = mo.forward_backward(net.get_params().astype(np.float64), net.layer_shapes(), x, t,
                                         round_bf16=True)
    assert abs(loss - loss_o) <= 2e-2 * loss_o
    assert np.linalg.norm(g - g_o) <= 2e-2 * np.linalg.norm(g_o)


def test_step_equals_adam_on_the_gradients():
    """A training step is Adam on exactly the gradients that sqh_mlp_gradients returns (the
    first step: m / c1 = g, v / c2 = g^2), and a smaller batch after a larger one reuses
    its buffers.  Bound: a few FP32 roundings of lr-sized updates."""
    ctx = Context(0)
    net = WarmStartMLP(ctx, 130, 192, 2, 70, seed=9)
    rng = np.random.default_rng(4)
    for B in (200, 65):
        twin = WarmStartMLP(ctx, 130, 192, 2, 70, seed=9)
        x = rng.standard_normal((B, 130)).astype(np.float32)
        t = rng.standard_normal((B, 70)).astype(np.float32)
        _, g = net.gradients(x, t)
        p = twin.get_params().astype(np.float64)
        xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        torch.cuda.synchronize()
        twin.train_step_dev(xd.data_ptr(), td.data_ptr(), B, 1e-3)
        g = g.astype(np.float64)
        want = p - 1e-3 * g / (np.abs(g) + 1e-8)
        np.testing.assert_allclose(twin.get_params(), want, rtol=0, atol=2e-6)
