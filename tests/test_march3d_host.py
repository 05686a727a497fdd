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
#include <vector>

#include "rsg_tiles3.h"
extern "C" {
unsigned off(int r, int nx, int c) { return rsg::tile_off(r, nx, c); }
int row0(int y0, int hy, int clip) { return rsg::window_row0(y0, hy, clip); }
int fit(int nx, int ny, int ty, int order) { return rsg::tiles_fit(nx, ny, ty, order); }

// The layout of a launch of ncomp components: out = {blocks, tx, zc, xgroups}.
void layout(const int *a, unsigned *out) {
    rsg::Tiles3 t;
    out[0] = rsg::layout_tiles3(t, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8]);
    out[1] = t.tx;
    out[2] = t.zc;
    out[3] = t.xgroups;
}

// The most blocks one XCD (r mod 8) holds, in percent of an eighth of all.
int share(const int *a) {
    rsg::Tiles3 t;
    const unsigned n = rsg::layout_tiles3(t, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8]);
    long live[8] = {}, all = 0;
    for (unsigned r = 0; r < n; r++) {
        rsg::Pos3 p{};
        const int l = t.tx == 64 ? rsg::tile3_at<64>(t, (int)r, p) : rsg::tile3_at<32>(t, (int)r, p);
        live[r % 8] += l;
        all += l;
    }
    return (int)(*std::max_element(live, live + 8) * 800 / all);
}

// Walks all blocks.  0: every plane of every tile is marched once a component,
// by a chunk that holds planes of one face's strip and shortened stencils or,
// in the middle zone, of none; else what is wrong.  kinds: bit 2 pxy + pz set
// where a block takes that instantiation.
int cover(const int *a, int *kinds) {
    const int nx = a[0], ny = a[1], nz = a[2], lpml = a[3], order = a[4], ncomp = a[5];
    rsg::Tiles3 t;
    const unsigned n = rsg::layout_tiles3(t, nx, ny, nz, lpml, order, ncomp, a[6], a[7], a[8]);
    const int ty = rsg::R3 * rsg::B3 / t.tx, m = std::max(lpml, order);
    std::vector<int> seen((size_t)t.ncx * t.ncy * nz * ncomp);
    *kinds = 0;
    for (unsigned r = 0; r < n; r++) {
        rsg::Pos3 p{};
        if (!(t.tx == 64 ? rsg::tile3_at<64>(t, (int)r, p) : rsg::tile3_at<32>(t, (int)r, p))) continue;
        if (p.x0 % t.tx || p.y0 % ty || p.x0 >= nx || p.y0 >= ny || p.comp < 0 || p.comp >= ncomp) return 1;
        if (p.zb < 0 || p.ze > nz || p.ze - p.zb > t.zc) return 2;
        for (int z = p.zb; z < p.ze; z++) {
            seen[(((size_t)z * t.ncy + p.y0 / ty) * t.ncx + p.x0 / t.tx) * ncomp + p.comp]++;
            if (p.zone == 1 && (z < m || z >= nz - m)) return 3;
            if (p.zone == 0 && z >= nz - lpml) return 4;
            if (p.zone == 2 && z < lpml) return 5;
        }
        *kinds |= 1 << (2 * rsg::tile_pxy(t.tx, nx, ny, lpml, order, p) + (p.zone != 1));
    }
    for (int s : seen)
        if (s != 1) return 6;
    return 0;
}
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


def _layout(m, *args):
    out = (C.c_uint * 4)()
    m.layout((C.c_int * 9)(*args), out)
    return dict(zip(("blocks", "tx", "zc", "xgroups"), out))


def test_every_plane_of_every_tile_is_marched_once(march):
    rng = random.Random(3)
    for i in range(400):
        order, lpml = rng.randint(1, 8), rng.randint(1, 20)
        n = [max(2 * lpml + 1, int(10 ** rng.uniform(0.5, 2.5))) for _ in range(3)]
        ncomp, first = rng.choice(((1, 0), (3, 0), (4, 1)))
        zc, xcd = rng.choice((0, 0, 1, 2, 3, 8, 16, 4096)), rng.randint(0, 1)
        a = (C.c_int * 9)(*n, lpml, order, ncomp, first, zc, xcd)
        kinds = C.c_int()
        assert march.cover(a, C.byref(kinds)) == 0, list(a)


def test_the_half_step_tests_reach_every_march(march):
    """The sizes the march is compared with the oracle at hold tiles and chunks
    with and without strips or shortened stencils, in both tile widths."""
    from tests.test_gpu_march3d import INNER, SIZES
    for ncomp in (1, 3, 4):
        kinds = {32: 0, 64: 0}
        for size in SIZES + INNER:
            a = (C.c_int * 9)(*size, ncomp, ncomp // 4, 0, 1)
            k = C.c_int()
            assert march.cover(a, C.byref(k)) == 0
            kinds[_layout(march, *a)["tx"]] |= k.value
        assert kinds == {32: 15, 64: 15}


# padded nx, ny, nz, lpml of small and of thin grids, and of one that fills the chip
@pytest.mark.parametrize("grid", [(24, 24, 24, 4), (32, 32, 32, 6), (48, 48, 48, 10), (64, 64, 64, 10), (70, 60, 50, 10),
                                  (20, 20, 400, 4), (400, 20, 20, 4), (20, 400, 20, 4), (33, 500, 33, 10),
                                  (140, 130, 120, 20)], ids=str)
def test_launches_spread_over_the_chip(march, grid):
    """No XCD gets more than an eighth above its share of the blocks, and an
    elastic launch whose blocks all run at once has chunks of one or two planes."""
    nx, ny, nz, lpml = grid
    for ncomp in (1, 3, 4):
        a = (nx, ny, nz, lpml, 4, ncomp, ncomp // 4, 0, 1)
        t = _layout(march, *a)
        assert t["blocks"] < 64 or march.share((C.c_int * 9)(*a)) <= 113, a
        if ncomp == 1:
            continue
        cols = -(-nx // t["tx"]) * -(-ny // (512 // t["tx"]))
        assert t["zc"] <= 2 or cols * ncomp * nz // 2 > 1000, t


# padded nx, ny, nz, components, zc3d: thin grids, and very large ones with
# short chunks asked for, whose blocks of 256 threads passed 2^32 threads
@pytest.mark.parametrize("nx,ny,nz,ncomp,zc", [(3, 8192, 65535, 4, 0), (3, 12000, 65535, 3, 0),
                                               (1300, 1300, 1300, 4, 1), (1400, 1400, 1400, 3, 1)])
def test_a_launch_holds_its_blocks(march, nx, ny, nz, ncomp, zc):
    for xcd in (0, 1):
        t = _layout(march, nx, ny, nz, 1, 8, ncomp, ncomp // 4, zc, xcd)
        assert 0 < t["blocks"] * 256 < 1 << 32, t


def _window_offsets(m, nx, ny, ty, order, clip=1):
    """(formed, exact) byte offsets of the corner cells of every distinct
    window: the first and last rows of tiles, the leftmost and rightmost."""
    for y0 in sorted({0, ty, 2 * ty, (ny - 1) // ty * ty}):
        if y0 >= ny:
            continue
        row0 = m.row0(y0, order, clip)
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


def test_acoustic_windows_fit_without_clipping(march):
    """Planes of up to 2^29 - 1 cells and at least 2 order + 2 rows, counted from
    the halo's corner."""
    rng = random.Random(5)
    grids = [(36_000_000, 14, 4), (89_000_000, 6, 2), (29_826_161, 18, 8)]
    for _ in range(300):
        order = rng.randint(1, 8)
        ny = rng.randint(2 * order + 2, 64)
        grids.append((((1 << 29) - 1) // ny, ny, order))
    for nx, ny, order in grids:
        assert nx * ny < 1 << 29
        for ty in (8, 16):
            for got, exact, at in _window_offsets(march, nx, ny, ty, order, 0):
                assert got == exact < KOUT, (nx, ny, order, at, got, exact)


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
