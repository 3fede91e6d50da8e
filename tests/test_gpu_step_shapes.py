"""GPU test of the automatic step shapes (the kernel without LDS on small
grids, the ring's tile shapes on larger ones) against the one-cell kernel:
partial groups, tiles and z chunks, every action, fields that reach the edges."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL = [(9, 9, 9), (10, 13, 11), (13, 10, 12), (45, 21, 19), (64, 35, 30), (131, 34, 29)]
LARGE = [(300, 220, 172), (388, 148, 196), (512, 145, 150)]  # > 10 M cells, n1 % 4 == 0


def _setup(dev, n, seed):
    r = np.random.default_rng(seed)
    n1, n2, n3 = n
    dev.create_space((10.0, 11.0, 12.0), 3.0, 0.01, n)
    dev.set_velocity(r.uniform(0.5, 8.0, n[::-1]).astype(np.float32))
    dev.set_imaging_scale(0.5)
    return r


def _both(dev, run):
    out = []
    try:
        for cells in (0, 1):
            dev.set_x_per_lane(cells)
            out.append(run())
    finally:
        dev.set_x_per_lane(0)
    return out


def _close(a, b):
    # the same operations in the same order per cell; only the order of the
    # imaging term's roundings and of contractions may differ
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert np.linalg.norm(b) > 0
    assert np.linalg.norm(a - b) <= 1e-6 * np.linalg.norm(b)


@pytest.mark.parametrize("n", SMALL + LARGE)
def test_plain_steps(dev, n):
    print(f"step shapes {n}", file=sys.stderr, flush=True)
    r = _setup(dev, n, 1)
    p = np.zeros((2,) + n[::-1], np.float32)
    p[:, 4:-4, 4:-4, 4:-4] = r.standard_normal((2, n[2] - 8, n[1] - 8, n[0] - 8))
    (a, ao), (b, bo) = _both(dev, lambda: dev.propagate(0, 3, p[0], p[1]))
    _close(a, b)
    _close(ao, bo)


@pytest.mark.parametrize("store", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("n", SMALL[3:] + LARGE[:2])
def test_shot_actions(dev, n, store):
    print(f"step shapes {n} {store}", file=sys.stderr, flush=True)
    r = _setup(dev, n, 2)
    n1, n2, n3 = n
    nt, ntr = 8, 16
    tab = np.zeros((1, 8), np.float32)
    tab[0, 3] = 1
    dev.set_sinc_table(0, tab)
    dev.set_sinc_table(1, tab)
    # source points all over the grid, receivers on every column of one plane
    npts = 300
    x, y, z = (r.integers(4, m - 4, npts) for m in (n1, n2, n3))
    locs = np.unique(x + y * n1 + z * n1 * n2).astype(np.int32)
    dev.set_source(locs, r.standard_normal((len(locs), ntr)).astype(np.float32))
    yy, xx = np.meshgrid(np.arange(n2), np.arange(n1), indexing="ij")
    rl = (xx + yy * n1 + (n3 // 2) * n1 * n2).astype(np.int32).ravel()
    data = r.standard_normal((len(rl), ntr)).astype(np.float32)
    model = r.standard_normal(n[::-1]).astype(np.float32)

    def run():
        dev.set_receivers(rl, data, nx=n1, ny=n2)
        dev.source_prop(1, nt, 1, store=store)
        dev.zero_image()
        dev.rtm_adjoint(1, nt, 1)
        img = dev.get_image()
        dev.set_model(model)
        dev.rtm_forward(1, nt, 1)
        return img, dev.get_receivers(), dev.get_snapshot(nt - 1)

    for a, b in zip(*_both(dev, run)):
        _close(a, b)
