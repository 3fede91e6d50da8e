"""GPU test of the network's gradients without rounding: integer inputs, weights
that pick one tap of one channel and a gradient that starts from single
positions at the tiles' edges, so that every sum is exact in FP32 whatever its
order and a product left out or counted twice anywhere shows.

Activations are multiples of 1/64 up to 1 (two averages of zeros and ones),
exact in BF16.  Gradients are multiples of 2 / (64 N), N positions a power of
two; where one needs more than BF16's eight bits before a layer's ReLU, the
reference rounds it there as the kernels do."""
import sys

import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu

EDGES = (0, 1, 3, 4, 7, 8, 15, 16, 17, 31, 32, 33, 47, 48, 55, 56, 62, 63)


def picks(r):
    """Parameters of a network whose output channels each copy one tap of one
    input channel; every input channel of a layer with no more inputs than
    outputs is used."""
    lay, n = U.layout()
    theta = np.zeros(n)
    for k, (ci, co) in enumerate([(1, 16)] + U.LAYERS):
        o, s = lay[f"w{k}"]
        w = theta[o:o + 27 * ci * co].reshape(27, co, ci)
        src = np.concatenate([r.permutation(ci) for _ in range(-(-co // ci))])[:co]
        w[r.integers(0, 27, co), np.arange(co), src] = 1.0
    o, s = lay["wh"]
    theta[o:o + 16] = r.choice((-1.0, 1.0), 16)
    return theta


def problem(batch, patch, seed, dtype=None):
    """theta, x, t, and the output and gradient of mean (net(x) - t)^2 by torch on
    the CPU."""
    import torch
    import torch.nn.functional as F
    dtype = dtype or torch.float32
    r = np.random.default_rng(seed)
    theta = picks(r)
    p = torch.from_numpy(theta).to(dtype).requires_grad_(True)
    lay, _ = U.layout()

    class RoundGrad(torch.autograd.Function):  # the gradient's BF16 rounding
        @staticmethod
        def forward(ctx, v):
            return v.view_as(v)

        @staticmethod
        def backward(ctx, g):
            return g.to(torch.float32).to(torch.bfloat16).to(dtype)

    def take(k):
        o, s = lay[k]
        return p[o:o + int(np.prod(s))].reshape(s)

    def conv(v, k):
        W = take(f"w{k}").reshape(27, -1, v.shape[1])
        W = W.permute(1, 2, 0).reshape(W.shape[1], W.shape[2], 3, 3, 3)
        return F.relu(RoundGrad.apply(F.conv3d(v, W, take(f"b{k}"), padding=1)))

    x = r.integers(0, 2, (batch,) + (patch,) * 3).astype(np.float32)
    X = torch.from_numpy(x).to(dtype)[:, None]
    s1 = conv(conv(X, 0), 1)
    s2 = conv(conv(F.avg_pool3d(s1, 2), 2), 3)
    y = conv(conv(F.avg_pool3d(s2, 2), 4), 5)
    y = conv(conv(torch.cat((F.interpolate(y, scale_factor=2), s2), 1), 6), 7)
    y = conv(conv(torch.cat((F.interpolate(y, scale_factor=2), s1), 1), 8), 9)
    out = X + F.conv3d(y, take("wh").reshape(1, 16, 1, 1, 1), take("bh"))
    # the residual: +-1 at positions where tiles, segments and planes meet
    e = np.zeros(x.shape, np.float32)
    edges = np.array([v + b for b in range(0, patch, 64) for v in EDGES])
    for n in range(batch):
        q = r.choice(edges, (300, 3))
        e[n, q[:, 0], q[:, 1], q[:, 2]] = r.choice((-1.0, 1.0), 300)
    o = out.detach().numpy()[:, 0]
    t = (o - e).astype(np.float32)
    (out - torch.from_numpy(t).to(dtype)[:, None]).square().mean().backward()
    return theta, x, t, o, p.grad.numpy()


@pytest.mark.parametrize("batch,patch", [(1, 64), (2, 64), (1, 128)])
def test_gradient_is_exact_on_integers(dev, batch, patch):
    from sep_code_amd.unet import UNet
    print(f"exact gradients {batch} x {patch}^3", file=sys.stderr, flush=True)
    theta, x, t, out, ref = problem(batch, patch, 5 + batch + patch)
    dev.create_space((10.0, 10.0, 10.0), 4.0, 0.0, (16, 16, 16))
    net = UNet(dev, batch=batch, patch=patch, seed=1)
    try:
        net.set_params(theta)
        np.testing.assert_array_equal(net.forward(x), out)
        _, g = net.loss_grad(x, t)
        lay, _ = U.layout()
        for k, (o, s) in lay.items():
            n = int(np.prod(s))
            assert np.count_nonzero(ref[o:o + n]) > 0, k
            np.testing.assert_array_equal(g[o:o + n], ref[o:o + n].astype(np.float32), k)
    finally:
        net.close()
