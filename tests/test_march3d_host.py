"""Host side of the 3D march, on the CPU: the index arithmetic of
csrc/rsg_tiles3.h (compiled alone with g++) against exact integers, and the
argument checks of the elastic 3D entries.  No GPU is needed."""
import ctypes as C
import os
import random
import subprocess

import pytest

from rockseis_amd import _lib as R

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rockseis_amd", "csrc")
KOUT = 0xFFFFFF00  # no descriptor covers offsets from here on

HARNESS = r"""
#include "rsg_tiles3.h"
extern "C" {
unsigned off(int r, int nx, int c) { return rsg::tile_off(r, nx, c); }
int row0(int y0, int hy) { return rsg::window_row0(y0, hy); }
int fit(int nx, int ny, int ty, int order) { return rsg::tiles_fit(nx, ny, ty, order); }
}
"""


@pytest.fixture(scope="module")
def march(tmp_path_factory):
    d = tmp_path_factory.mktemp("march3d")
    src, so = d / "march.cpp", d / "march.so"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o",
                    str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.off.restype = C.c_uint
    return lib


def _window_offsets(m, nx, ny, ty, order):
    """(formed, exact) byte offsets of the corner cells of every distinct
    window: the first and last rows of tiles, the leftmost and rightmost."""
    for y0 in sorted({0, ty, 2 * ty, (ny - 1) // ty * ty}):
        if y0 >= ny:
            continue
        row0 = m.row0(y0, order)
        for y in {max(y0 - order, 0), y0, min(y0 + ty + order, ny) - 1}:
            for x0 in {0, (nx - 1) // 64 * 64}:
                for x in {max(x0 - order, 0), min(x0 + 64 + order, nx) - 1}:
                    c = x - (x0 - order)
                    yield m.off(y - row0, nx, c), ((y - row0) * nx + c) * 4, (x0, y0, x, y)


# acoustic planes (< 2^29 cells) and elastic ones whose windows reach past
# 2^31 bytes counted from the halo's corner: order 4, 8, 2, 8, 8, 1
WIDE = [(36_000_000, 14, 4), (30_000_000, 17, 8), (89_000_000, 6, 2), (1 << 25, 12, 8), (44_000_000, 200, 8),
        (100_000_000, 10, 1)]


@pytest.mark.parametrize("nx,ny,order", WIDE)
def test_window_offsets_of_long_rows(march, nx, ny, order):
    assert march.fit(nx, ny, 8, order)
    for got, exact, at in _window_offsets(march, nx, ny, 8, order):
        assert got == exact < KOUT, (at, got, exact)


def test_tiles_fit_says_where_offsets_end(march):
    rng = random.Random(7)
    seen = set()
    for _ in range(4000):
        order, ty = rng.randint(1, 8), rng.choice((8, 16))
        ny, nx = rng.randint(3, 60), int(10 ** rng.uniform(1, 8.7))
        worst = max(e for _, e, _ in _window_offsets(march, nx, ny, ty, order))
        fit = bool(march.fit(nx, ny, ty, order))
        seen.add(fit)
        if fit:  # every offset formed is exact and covered
            assert worst + 4 <= KOUT, (nx, ny, ty, order)
            assert all(g == e for g, e, _ in _window_offsets(march, nx, ny, ty, order))
        else:    # and no grid is refused that lies well inside
            assert min(ny, ty + 2 * order) * nx * 4 > KOUT - 64, (nx, ny, ty, order)
    assert seen == {False, True}


def _e3d(nx, ny, nz, order):
    g = R.Grid(nx=nx, ny=ny, nz=nz, lpml=1, order=order, fs=0, dx=10, dy=10, dz=10, dt=1e-3)
    s = R.StateE3D()
    for n, _ in R.StateE3D._fields_[:-1]:
        setattr(s, n, 1 << 12)
    for i in range(R.E3D_NSTRIP):
        s.psi[i] = 1 << 12
    return g, s


def test_sources_and_receivers_take_grids_of_any_width():
    """Injection and gathers use 64-bit indices: no limit of the march's
    windows applies to them (no trace: nothing is launched)."""
    lib = R.lib()
    none = R.Traces(R.PRESSURE, 0, 1, None, None, None, None)
    for nx, ny in ((1 << 24, 40), (1 << 26, 17)):
        g, s = _e3d(nx, ny, 3, 8)
        assert lib.rsg_e3d_insert_source(C.byref(g), C.byref(s), C.byref(none), 0, None) == 0, lib.rsg_last_error()
        assert lib.rsg_e3d_record_data(C.byref(g), C.byref(s), C.byref(none), None, None, None, 0, None) == 0, \
            lib.rsg_last_error()


def test_steps_refuse_rows_past_32_bit_offsets():
    lib = R.lib()
    g, s = _e3d(1 << 26, 17, 3, 8)  # 17 rows of 2^28 bytes
    for f in (lib.rsg_e3d_forward_velocity, lib.rsg_e3d_forward_stress, lib.rsg_e3d_backward_stress):
        assert f(C.byref(g), C.byref(s), None) == -1
        assert b"32-bit offsets" in lib.rsg_last_error()
    assert lib.rsg_e3d_backward_velocity_ws(C.byref(g), C.byref(s), C.c_void_p(1 << 12), None) == -1
    assert b"32-bit offsets" in lib.rsg_last_error()
