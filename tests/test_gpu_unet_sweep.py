"""GPU test of the network where its convolutions are cut differently: the
planes per sweep depend on the batch, the result of a patch must not."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("patch,batches", [(64, (1, 2, 5, 16)), (128, (1, 3))])
def test_output_does_not_depend_on_the_batch(dev, patch, batches):
    from sep_code_amd.unet import UNet
    dev.create_space((10.0, 10.0, 10.0), 4.0, 0.0, (16, 16, 16))
    net = UNet(dev, batch=max(batches), patch=patch, seed=5)
    theta = net.get_params()
    theta[-17:] = np.linspace(-0.5, 0.5, 17)  # the head: every channel reaches the output
    net.set_params(theta)
    r = np.random.default_rng(patch)
    x = r.standard_normal((max(batches),) + (patch,) * 3).astype(np.float32)
    ref = {}
    for nb in batches:
        print(f"sweep patch {patch} batch {nb}", file=sys.stderr, flush=True)
        y = net.forward(x[:nb])
        assert np.isfinite(y).all() and np.std(y - x[:nb]) > 0
        for k in range(nb):
            assert np.array_equal(y[k], ref.setdefault(k, y[k])), (nb, k)
    net.close()


@pytest.mark.parametrize("channel,batch", [(0, 1), (7, 3), (15, 2)])
def test_head_gradient(dev, channel, batch):
    """With one head weight 1 and the rest 0 the output shows that channel."""
    from sep_code_amd.unet import UNet
    dev.create_space((10.0, 10.0, 10.0), 4.0, 0.0, (16, 16, 16))
    net = UNet(dev, batch=batch, patch=64, seed=9)
    theta = net.get_params()
    theta[-17:] = 0
    theta[-17 + channel] = 1
    net.set_params(theta)
    r = np.random.default_rng(channel)
    x = r.standard_normal((batch, 64, 64, 64)).astype(np.float32)
    t = r.standard_normal(x.shape).astype(np.float32)
    out = net.forward(x).astype(np.float64)
    _, g = net.loss_grad(x, t)
    _, g2 = net.loss_grad(x, t)
    assert np.array_equal(g[-17:], g2[-17:])  # partial sums added in a fixed order
    d = 2.0 / x.size * (out - t)
    for got, terms in ((g[-17 + channel], d * (out - x)), (g[-1], d)):
        # FP32 sums: far below 1e-5 of the terms' absolute sum
        assert abs(got - terms.sum()) <= 1e-5 * np.abs(terms).sum()
    net.close()
