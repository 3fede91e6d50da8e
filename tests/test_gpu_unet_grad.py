"""GPU test of the network's gradients where the work is cut differently:
batches (units per workgroup), a patch two row segments wide, and repeated
runs (the partial sums are added in a fixed order)."""
import sys

import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu


def _net(dev, batch, patch, seed):
    from sep_code_amd.unet import UNet
    dev.create_space((10.0, 10.0, 10.0), 4.0, 0.0, (16, 16, 16))
    net = UNet(dev, batch=batch, patch=patch, seed=seed)
    theta = net.get_params().astype(np.float64)
    lay, _ = U.layout()
    r = np.random.default_rng(seed)
    for k, (o, s) in lay.items():
        n = int(np.prod(s))
        if k == "wh":
            theta[o:o + n] = 0.5 * r.standard_normal(n)
        elif k.startswith("b"):
            theta[o:o + n] = 0.05 * r.standard_normal(n)
    net.set_params(theta)
    return net


def _reference_grad(theta, x, t):
    """Gradient of mean (net(x) - t)^2 by torch autograd on the CPU in FP32."""
    import torch
    import torch.nn.functional as F
    p = torch.from_numpy(theta.astype(np.float32)).requires_grad_(True)
    lay, _ = U.layout()

    def take(k):
        o, s = lay[k]
        return p[o:o + int(np.prod(s))].reshape(s)

    def conv(v, k):
        W = take(f"w{k}").reshape(27, -1, v.shape[1])
        W = W.permute(1, 2, 0).reshape(W.shape[1], W.shape[2], 3, 3, 3)
        return F.relu(F.conv3d(v, W, take(f"b{k}"), padding=1))

    X = torch.from_numpy(x)[:, None]
    s1 = conv(conv(X, 0), 1)
    s2 = conv(conv(F.avg_pool3d(s1, 2), 2), 3)
    y = conv(conv(F.avg_pool3d(s2, 2), 4), 5)
    y = conv(conv(torch.cat((F.interpolate(y, scale_factor=2), s2), 1), 6), 7)
    y = conv(conv(torch.cat((F.interpolate(y, scale_factor=2), s1), 1), 8), 9)
    out = X + F.conv3d(y, take("wh").reshape(1, 16, 1, 1, 1), take("bh"))
    (out - torch.from_numpy(t)[:, None]).square().mean().backward()
    return p.grad.numpy()


@pytest.mark.parametrize("batch,patch", [(1, 64), (3, 64), (1, 128)])
def test_gradient_against_torch_and_repeatable(dev, batch, patch):
    net = _net(dev, batch, patch, 7 + batch)
    r = np.random.default_rng(patch + batch)
    x = r.standard_normal((batch, patch, patch, patch)).astype(np.float32)
    t = r.standard_normal(x.shape).astype(np.float32)
    _, g = net.loss_grad(x, t)
    _, g2 = net.loss_grad(x, t)
    lay, _ = U.layout()
    head = set(range(lay["wh"][0], lay["bh"][0] + 1))
    same = g == g2
    assert all(same[i] or i in head for i in range(g.size))
    ref = _reference_grad(net.get_params(), x, t)
    for k, (o, s) in lay.items():
        if k in ("wh", "bh"):
            continue  # the head's gradient has its own kernel (and bh's sum cancels)
        n = int(np.prod(s))
        e = np.linalg.norm(g[o:o + n] - ref[o:o + n]) / np.linalg.norm(ref[o:o + n])
        print(f"  batch {batch} patch {patch} grad {k}: {e:.3e}", file=sys.stderr, flush=True)
        # BF16 activations and weights through up to ten layers: the bar of
        # the network's own oracle test
        assert e < 8e-2, k
    net.close()
