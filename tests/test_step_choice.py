"""CPU test of the rule that chooses a time step's kernel and tile shape
(sep_code_amd/csrc/step_choice.h, built here with g++ on its own)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PLAIN, IMG, BORN = 0, 1, 2
F32, F16 = 1, 3
NONE, INJECT, EXTRACT = 0, 1, 2

SRC = """
#include <cstring>
#include "step_choice.h"
using namespace brtm;
extern "C" void choose(const int *s, int form, int act, int fmt, int rec, int *out, char *name) {
  const StepSetting S{s[0], s[1], s[2], 256, s[3], 2048, s[4], s[5]};
  const StepChoice c = choose_step(S, form, act, fmt, rec);
  const int v[8] = {c.kernel, c.tw, c.ty, c.zc, c.ntx, c.nty, c.ntz, c.rec};
  std::memcpy(out, v, sizeof(v));
  std::strcpy(name, step_kernel_name(c).c_str());
}
"""


@pytest.fixture(scope="session")
def choose(tmp_path_factory):
    d = tmp_path_factory.mktemp("choice")
    (d / "c.cpp").write_text(SRC)
    so = d / "libc.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "sep_code_amd", "csrc"), "-o", str(so), str(d / "c.cpp")],
                   check=True)
    lib = C.CDLL(str(so))

    def run(n, act=PLAIN, fmt=0, rec=NONE, form=0, ty=0, xl=0, ring=-1):
        out, name = (C.c_int * 8)(), C.create_string_buffer(128)
        lib.choose((C.c_int * 6)(*n, ty, xl, ring), form, act, fmt, rec, out, name)
        return name.value.decode().replace(" (", ",").split(",")[0], list(out), name.value.decode()

    return run


@pytest.mark.parametrize("n,act,fmt,kernel,tile", [
    ((48, 48, 48), PLAIN, 0, "k_step_direct", 1),
    ((128, 128, 128), PLAIN, 0, "k_step_direct", 2),
    ((131, 131, 131), IMG, F16, "k_step_direct", 2),
    ((256, 256, 256), PLAIN, 0, "k_step_x4r", (256, 8)),
    ((256, 256, 256), BORN, F16, "k_step_x4r", (256, 8)),
    ((512, 512, 512), PLAIN, 0, "k_step_x4r", (256, 16)),
    ((512, 512, 512), IMG, F32, "k_step_x4r", (256, 8)),
    ((288, 240, 208), PLAIN, 0, "k_step_x4r", (64, 16)),
    ((384, 384, 384), PLAIN, 0, "k_step_x4r", (128, 24)),
    ((302, 302, 302), PLAIN, 0, "k_step_x2", (128, 16)),
    ((301, 301, 301), PLAIN, 0, "k_step", (64, 32)),
])
def test_automatic_kernels(choose, n, act, fmt, kernel, tile):
    got, c, name = choose(n, act, fmt)
    assert got == kernel, name
    assert (c[3] if kernel == "k_step_direct" else (c[1], c[2])) == tile, name


def test_extracting_steps_take_taller_tiles(choose):
    """Plain steps of Born modelling, which extract receivers, run in 16-row
    tiles at 256^3, where the others take 8 rows; steps with an action keep
    their shape."""
    n = (256, 256, 256)
    assert choose(n, rec=EXTRACT)[1][1:3] == [256, 16]
    assert choose(n, rec=INJECT)[1][1:3] == choose(n)[1][1:3] == [256, 8]
    assert choose(n, BORN, F16, EXTRACT)[1][1:3] == choose(n, BORN, F16)[1][1:3] == [256, 8]


@pytest.mark.parametrize("n,act,fmt,want", [
    # grids where 64 x 16 tiles, or the kernel without LDS (plain steps below
    # 10 M cells), were slower than the one- and two-cell kernels
    ((164, 544, 393), IMG, F32, "256x8 tiles"), ((164, 544, 393), IMG, F16, "256x8 tiles"),
    ((564, 293, 259), IMG, F32, "256x8 tiles"), ((264, 368, 128), IMG, F16, "no LDS"),
    ((300, 220, 172), IMG, F32, "no LDS"), ((272, 541, 86), IMG, F16, "no LDS"),
    ((164, 294, 237), IMG, F32, "no LDS"), ((204, 248, 235), PLAIN, 0, "256x16 tiles"),
    ((196, 248, 213), PLAIN, 0, "256x16 tiles"), ((224, 256, 160), PLAIN, 0, "256x8 tiles"),
])
def test_grids_that_narrow_tiles_fit_badly(choose, n, act, fmt, want):
    assert want in choose(n, act, fmt)[2]


@pytest.mark.parametrize("xl,ring,ty,kernel,tile", [
    (1, -1, 0, "k_step", (64, 32)), (1, 1, 16, "k_step_ring", (64, 16)),
    (2, -1, 0, "k_step_x2", (128, 16)), (4, 0, 0, "k_step_x4", (256, 16)),
    (4, 1, 8, "k_step_x4r", (256, 8)), (4, -1, 32, "k_step_x4r", (256, 16)),
    (0, -1, 8, "k_step_x4r", (256, 8)), (0, 0, 0, "k_step_x4", (256, 16)),
])
def test_settings_keep_their_kernels(choose, xl, ring, ty, kernel, tile):
    got, c, name = choose((256, 128, 128), xl=xl, ring=ring, ty=ty)
    assert got == kernel and (c[1], c[2]) == tile, name
    # the LV form has only the one-cell tiles
    assert choose((256, 128, 128), form=1, xl=xl, ring=ring, ty=ty)[0] == "k_step"


def test_chunks_cover_the_update_set(choose):
    """Tiles and z chunks of every choice cover the grid once, no chunk empty,
    and a step that takes receivers inside says so."""
    for n1 in (9, 12, 45, 64, 130, 131, 257, 320, 512, 1000):
        for n2 in (9, 64, 131, 300):
            for n3 in (9, 10, 65, 200, 400):
                for act, fmt in ((PLAIN, 0), (IMG, F32), (IMG, F16), (BORN, F16)):
                    for xl in (0, 1, 2, 4):
                        got, c, name = choose((n1, n2, n3), act, fmt, EXTRACT, xl=xl)
                        _, tw, ty, zc, ntx, nty, ntz, rec = c
                        what = ((n1, n2, n3), act, fmt, xl, name)
                        nz = n3 - 8
                        assert zc >= 1 and (ntz - 1) * zc < nz <= ntz * zc, what
                        if got == "k_step_direct":
                            groups = (n1 - 5) // 4 * (n2 - 8)
                            assert 256 * (ntx - 1) < groups <= 256 * ntx, what
                        else:
                            assert (ntx - 1) * tw < n1 <= ntx * tw, what
                            assert (nty - 1) * ty < n2 <= nty * ty, what
                        assert (rec == EXTRACT) == (got in ("k_step_direct", "k_step_x4r") or
                                                    (got == "k_step" and ty == 8)), what
