"""GPU test of the kernels that only larger or particular grids reach (two z
slices per thread without LDS; the ring's 128 x 24, 64 x 16 and 256 x 16
tiles, with and without streaming loads) against the one-cell kernel, each
named by the library; and of the benchmark's label."""
import os
import sys

import numpy as np
import pytest

from test_gpu_step_shapes import _both, _close, _setup

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DIRECT2 = "k_step_direct (4 cells/lane, no LDS), 2 slices per thread"


def _ring(tiles):
    return f"k_step_x4r (4 cells/lane, six-plane halo ring), {tiles} tiles"


# (grid, streaming loads, kernel of plain steps, of steps with an action)
GRIDS = [
    # the last z chunk half empty; rows that end in a group of 3, 2 and 4 cells
    ((147, 122, 133), -1, DIRECT2, DIRECT2),
    ((150, 121, 131), -1, DIRECT2, DIRECT2),
    ((128, 131, 133), -1, DIRECT2, DIRECT2),
    # partial tiles in x, y and z
    ((380, 284, 104), 0, _ring("128x24"), _ring("128x24")),
    ((380, 284, 104), 1, _ring("128x24"), _ring("128x24")),
    ((304, 220, 200), 0, _ring("64x16"), _ring("64x16")),
    ((304, 220, 200), 1, _ring("64x16"), _ring("64x16")),
    ((508, 218, 132), 0, _ring("256x16"), _ring("256x8")),
    ((508, 218, 132), 1, _ring("256x16"), _ring("256x8")),
]


def _names(dev, stream, plain, action):
    end = " + streaming loads" if stream == 1 else ""
    assert all(dev.step_kernel(0, 0, 0, rec) == plain + end for rec in (0, 1, 2))
    for act, rec in ((1, 1), (2, 2)):
        for fmt in (1, 2, 3):
            assert dev.step_kernel(0, act, fmt, rec) == action + end


@pytest.mark.parametrize("store", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("n,stream,plain,action", GRIDS)
def test_shots_on_the_larger_kernels(dev, n, stream, plain, action, store):
    print(f"step kernels {n} stream {stream} {store}", file=sys.stderr, flush=True)
    r = _setup(dev, n, 11)
    n1, n2, n3 = n
    nt, ntr = 4, 12
    tab = np.zeros((1, 8), np.float32)
    tab[0, 3] = 1
    dev.set_sinc_table(0, tab)
    dev.set_sinc_table(1, tab)
    npts = 300  # source points all over the grid
    x, y, z = (r.integers(4, m - 4, npts) for m in (n1, n2, n3))
    locs = np.unique(x + y * n1 + z * n1 * n2).astype(np.int32)
    dev.set_source(locs, r.standard_normal((len(locs), ntr)).astype(np.float32))
    # receivers on every column of the last plane of the update set
    yy, xx = np.meshgrid(np.arange(n2), np.arange(n1), indexing="ij")
    rl = (xx + yy * n1 + (n3 - 5) * n1 * n2).astype(np.int32).ravel()
    data = r.standard_normal((len(rl), ntr)).astype(np.float32)
    model = r.standard_normal(n[::-1], dtype=np.float32)
    p = np.zeros((2,) + n[::-1], np.float32)
    p[:, 4:-4, 4:-4, 4:-4] = r.standard_normal((2, n3 - 8, n2 - 8, n1 - 8), dtype=np.float32)

    def run():
        a, b = dev.propagate(0, 2, p[0], p[1])
        dev.set_receivers(rl, data, nx=n1, ny=n2)
        dev.source_prop(1, nt, 1, store=store)
        dev.zero_image()
        dev.rtm_adjoint(1, nt, 1)
        img = dev.get_image()
        dev.set_model(model)
        dev.rtm_forward(1, nt, 1)
        return a, b, img, dev.get_receivers(), dev.get_snapshot(nt - 1)

    try:
        dev.set_stream_loads(stream)
        _names(dev, stream, plain, action)
        for a, b in zip(*_both(dev, run)):
            _close(a, b)
    finally:
        dev.set_stream_loads(-1)


@pytest.mark.parametrize("store", ["f32", "f16"])
@pytest.mark.parametrize("n", [(53, 44, 40), (131, 37, 29)])
def test_one_cell_tiles_with_receivers_inside(dev, n, store):
    """The one-cell step's 64 x 8 tiles, which take receivers inside the step:
    traces bit-identical to the separate extraction, images to FP32 rounding
    of the separate injection."""
    print(f"one-cell tiles {n} {store}", file=sys.stderr, flush=True)
    r = _setup(dev, n, 12)
    n1, n2, n3 = n
    nt, ntr = 6, 14
    tab = np.zeros((1, 8), np.float32)
    tab[0, 3] = 1
    dev.set_sinc_table(0, tab)
    dev.set_sinc_table(1, tab)
    dev.set_source(np.array([n1 // 2 + n1 * (n2 // 2) + n1 * n2 * (n3 // 2)], np.int32),
                   r.standard_normal((1, ntr)).astype(np.float32))
    yy, xx = np.meshgrid(np.arange(n2), np.arange(n1), indexing="ij")
    rl = (xx + yy * n1 + 4 * n1 * n2).astype(np.int32).ravel()
    data = r.standard_normal((len(rl), ntr)).astype(np.float32)
    model = r.standard_normal(n[::-1]).astype(np.float32)
    out = []
    try:
        dev.set_x_per_lane(1)
        dev.set_tuning(8, 2048)
        assert dev.step_kernel(0, 1, 1, 1) == "k_step, 64x8 tiles"
        for fuse in (0, 1):
            dev.set_receiver_fusion(fuse)
            dev.set_receivers(rl, data, nx=n1, ny=n2)
            dev.source_prop(1, nt, 1, store=store)
            dev.zero_image()
            dev.rtm_adjoint(1, nt, 1)
            img = dev.get_image()
            dev.set_model(model)
            dev.rtm_forward(1, nt, 1)
            out.append((img, dev.get_receivers()))
    finally:
        dev.set_receiver_fusion(1)
        dev.set_tuning(0, 2048)
        dev.set_x_per_lane(0)
    np.testing.assert_array_equal(out[1][1], out[0][1])
    _close(out[1][0], out[0][0])


@pytest.mark.parametrize("n,kernel", [((128, 128, 128), "k_step_direct"),
                                      ((288, 240, 208), "64x16 tiles"),
                                      ((512, 218, 132), "256x16 tiles")])
def test_benchmark_label_is_the_kernel_that_runs(dev, n, kernel):
    """bench.py names what the library chooses, not a copy of its rule."""
    sys.path.insert(0, ROOT)
    import bench
    dev.create_space((10.0, 10.0, 10.0), 3.0, 0.01, n)
    label = bench.plain_step_label(dev)
    assert label.startswith("brtm::" + dev.step_kernel(0, 0, 0, 1)) and kernel in label
