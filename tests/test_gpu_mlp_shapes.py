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


def _chain(values):
    s = np.float32(0)
    for v in values:
        s = np.float32(s + np.float32(v))
    return s


# one nonzero per 32-wide step of the sum: what is added to 2^25 before it is taken away again is
# lost, and only then, in one sum in ascending order
STEPS = [2.0 ** 25, 1, 1, 1, -2.0 ** 25, 3, 3, 3]


@pytest.mark.parametrize("rows,cols", [(64, 64), (1024, 1024)])  # 32 x 32 and 64 x 64 tiles
def test_products_are_one_sum_in_ascending_k(rows, cols):
    print(rows, cols, flush=True)
    K = 32 * len(STEPS)
    net = WarmStartMLP(Context(0), K, 1, 0, cols, seed=1)
    net.set_params(np.concatenate([np.ones(cols * K), np.zeros(cols)]).astype(np.float32))
    x = np.zeros((rows, K), dtype=np.float32)
    x[:, ::32] = STEPS
    xd, yd = torch.from_numpy(x).cuda(), torch.empty((rows, cols), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    net.forward_dev(xd.data_ptr(), rows, yd.data_ptr())
    net.ctx.synchronize()
    assert np.all(yd.cpu().numpy() == _chain(STEPS))


@pytest.mark.parametrize("ind,out", [(64, 64), (1024, 1024)])
def test_gradients_are_one_sum_over_the_batch(ind, out):
    """The weight gradient is one sum in ascending samples; the bias gradient is 64 slices
    (samples s, s + 64, ...), then the slices in order."""
    print(ind, out, flush=True)
    B = 32 * len(STEPS)
    net = WarmStartMLP(Context(0), ind, 1, 0, out, seed=1)
    net.set_params(np.zeros(out * ind + out, dtype=np.float32))
    t = np.zeros((B, out), dtype=np.float32)
    t[::32] = -np.asarray(STEPS)[:, None] * (B * out / 2)  # dY = 2 (0 - t) / (B out), exactly
    _, g = net.gradients(np.ones((B, ind), dtype=np.float32), t)
    assert np.all(g[:out * ind] == _chain(STEPS))
    assert np.all(g[out * ind:] == _chain([_chain(STEPS[0::2]), _chain(STEPS[1::2])]))


def test_adam_roundings():
    """An update is, in FP32: m <- fma(1 - b1, g, b1 m), v <- fma((1 - b2) g, g, b2 v),
    w <- w - lr (m / c1) / (sqrt(v / c2) + eps), each operation rounded once."""
    import ctypes
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    F = np.float32
    fma = lambda a, b, c: (a.astype(np.longdouble) * b + c).astype(F)  # noqa: E731  (products are exact)
    net = WarmStartMLP(Context(0), 65, 63, 1, 40, seed=3)
    rng = np.random.default_rng(8)
    b1, b2, lr = F(0.9), F(0.999), F(1e-3)
    w = net.get_params()
    m, v = np.zeros_like(w), np.zeros_like(w)
    for k in range(1, 5):
        x = rng.standard_normal((100, 65)).astype(F)
        t = rng.standard_normal((100, 40)).astype(F)
        _, g = net.gradients(x, t)
        xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        torch.cuda.synchronize()
        net.train_step_dev(xd.data_ptr(), td.data_ptr(), 100, float(lr))
        m = fma(np.full_like(g, F(1) - b1), g, b1 * m)
        v = fma((F(1) - b2) * g, g, b2 * v)
        c1, c2 = F(1) - F(powf(b1, k)), F(1) - F(powf(b2, k))
        w = w - lr * (m / c1) / (np.sqrt(v / c2) + F(1e-8))
        assert np.array_equal(net.get_params(), w)
