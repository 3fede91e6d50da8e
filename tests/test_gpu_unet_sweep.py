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
