"""CPU test of how the network's convolutions are cut for a device
(sep_code_amd/csrc/conv_plan.h, built here with g++ on its own)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "p.cpp").write_text(
        '#include "conv_plan.h"\n'
        'extern "C" int planes(long t, int d, int n, int c) { return brtm::sweep_planes(t, d, n, c); }\n'
        'extern "C" int groups(long u, int c, int w, long m) { return brtm::grad_groups(u, c, w, m); }\n')
    so = d / "libp.so"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "sep_code_amd", "csrc"), "-o", str(so), str(d / "p.cpp")],
                   check=True)
    lib = C.CDLL(str(so))
    lib.planes.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int]
    lib.groups.argtypes = [C.c_long, C.c_int, C.c_int, C.c_long]
    return lib


def test_sweeps_fill_the_device_that_there_is(plan):
    # 32 tiles of eight waves
    assert plan.planes(8 * 4, 64, 512, 256) == 8
    # a device of an eighth of the compute units sweeps further
    assert plan.planes(8 * 4, 64, 512, 32) == 16
    for depth in (16, 32, 48, 64, 80, 128):
        for tiles in (1, 4, 15, 64, 1000):
            for threads in (64, 256, 512):
                for ncu in (32, 64, 256, 304):
                    zl = plan.planes(tiles, depth, threads, ncu)
                    assert 1 <= zl <= 16 and depth % zl == 0
                    want = ncu if threads > 256 else 2 * ncu
                    assert zl == 1 or tiles * (depth // zl) >= want


def test_weight_gradients_fill_the_device_that_there_is(plan):
    most = (8 << 20) // (27 * 16 * 16 + 16)
    assert plan.groups(4 * 64 * 8, 256, 3, most) == 256
    assert plan.groups(4 * 64 * 8, 32, 3, most) == 32
    assert plan.groups(4 * 16 * 2, 256, 1, 75) == 75    # scratch for 75 partials
    assert plan.groups(16 * 2, 256, 2, 1000) == 32      # the volume's units
    assert plan.groups(5, 2, 1, 100) == 1               # never none
