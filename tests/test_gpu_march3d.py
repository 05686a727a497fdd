"""The 3D z march (rsg_fd3d.h) against the FP32 oracle on random states: one
velocity and one stress half step (acoustic; elastic, and its adjoint state's)
at the sizes where a tile, a chunk or a
strip can go wrong (rows of 64 and of 32, one cell more and less, strips
thinner than the stencil, chunks of odd length, tiles and chunks with no strip
or shortened stencil at all), every stencil order.

Moduli of about 1e4 make dt M / dx about one, so that what a step adds is as
large as the field it is added to: one cell of 10^5 off by 0.3% of the field, or
a coefficient off by 2e-5, shows.

Bound: an updated cell is a sum of up to 3 (2 order + 3) products; with
|terms| about four times the result in the 2-norm of a random state, two
orders of summing them differ by at most 4 * 57 / 2 units of 2^-24, 7e-6."""
import ctypes as C

import numpy as np
import pytest

from tests.gpu_util import RTOL_L2, rel_l2

pytestmark = pytest.mark.gpu

# padded nx, ny, nz, lpml, order
SIZES = [(64, 16, 12, 1, 1), (65, 17, 13, 2, 2), (40, 40, 90, 6, 3), (160, 50, 37, 18, 4), (97, 35, 29, 12, 4),
         (63, 64, 41, 4, 5), (31, 18, 18, 5, 6), (66, 22, 26, 10, 7), (33, 19, 23, 3, 8), (128, 24, 40, 9, 8)]
# with tiles inside all strips, of 32 x 16, 32 x 16 and 64 x 8 cells
INNER = [(80, 56, 40, 8, 8), (136, 40, 40, 6, 5), (192, 40, 30, 10, 4)]
# the elastic steps also take grids shorter than the stencil
SHORT = [(9, 7, 8, 2, 8), (20, 70, 5, 1, 4)]

E3D_MODEL = ("L", "L2M", "Mxz", "Myz", "Mxy", "Rx", "Ry", "Rz")


def _random(rng, *arrays):
    for a in arrays:
        a[...] = rng.standard_normal(a.shape)


def _moduli(rng, size, n):
    nx, ny, nz = size[:3]
    return [rng.uniform(0.5e4, 1.5e4, (nz, ny, nx)).astype(np.float32) for _ in range(n)]


def _compare(name, got, want):
    e = rel_l2(got, want)
    assert e <= RTOL_L2, f"{name}: rel L2 {e:.2e}"


class _A3D:
    """A random acoustic state in the oracle; step() takes both half steps of a
    copy on the device and returns its fields and strips."""
    fields = ("P", "Vx", "Vy", "Vz")

    def __init__(self, size):
        from oracle import runs
        self.size = size
        rng = np.random.default_rng(sum(size))
        self.o = o = runs.A3DState(*_moduli(rng, size, 4), *size[3:], 10.0, 12.5, 8.0, 1.5e-3)
        _random(rng, o.P, o.Vx, o.Vy, o.Vz, *o.strips.values())
        self.names = self.fields + tuple(o.strips)

    def step(self):
        import torch
        from rockseis_amd import _lib as R
        nx, ny, nz, lpml, order = self.size
        o = self.o
        dev = {k: torch.from_numpy(getattr(o, k).copy()).cuda() for k in self.fields + ("L", "Rx", "Ry", "Rz", "tab")}
        dev.update({k: torch.from_numpy(a.copy()).cuda() for k, a in o.strips.items()})
        g = R.Grid(nx=nx, ny=ny, nz=nz, lpml=lpml, order=order, fs=0, dx=10.0, dy=12.5, dz=8.0, dt=1.5e-3)
        s = R.State()
        for k in self.fields + ("L", "Rx", "Ry", "Rz", "tab"):
            setattr(s, k, dev[k].data_ptr())
        for i, k in enumerate(R.A3D_STRIPS):
            s.psi[i] = dev[k].data_ptr()
        st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        print(f"a3d {self.size}", flush=True)
        R.check(R.lib().rsg_a3d_forward_velocity(C.byref(g), C.byref(s), st), "velocity")
        R.check(R.lib().rsg_a3d_forward_stress(C.byref(g), C.byref(s), st), "stress")
        return [dev[k].cpu().numpy() for k in self.names]

    def expect(self):
        self.o.velocity()
        self.o.stress()
        return [getattr(self.o, k) for k in self.fields] + list(self.o.strips.values())


class _E3D:
    """The same for an elastic state and its forward or adjoint-state steps."""

    def __init__(self, size, adjoint):
        from oracle import runs
        self.size, self.adjoint = size, adjoint
        self.fields = runs.E3D_FIELDS
        self.fs = size[4] % 2
        rng = np.random.default_rng(sum(size))
        self.o = o = runs.E3DState(_moduli(rng, size, len(E3D_MODEL)), *size[3:], (10.0, 12.5, 8.0), 1.5e-3, self.fs)
        _random(rng, *(getattr(o, k) for k in self.fields), *o.strips)
        self.names = self.fields + tuple(f"strip {i}" for i in range(len(o.strips)))

    def step(self):
        import torch
        from rockseis_amd import _lib as R
        nx, ny, nz, lpml, order = self.size
        o = self.o
        dev = {k: torch.from_numpy(getattr(o, k).copy()).cuda() for k in self.fields + E3D_MODEL + ("tab",)}
        strips = [torch.from_numpy(a.copy()).cuda() for a in o.strips]
        g = R.Grid(nx=nx, ny=ny, nz=nz, lpml=lpml, order=order, fs=self.fs, dx=10.0, dy=12.5, dz=8.0, dt=1.5e-3)
        s = R.StateE3D()
        for k, t in dev.items():
            setattr(s, k, t.data_ptr())
        for i, t in enumerate(strips):
            s.psi[i] = t.data_ptr()
        st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        lib = R.lib()
        print(f"e3d {self.size} adjoint {self.adjoint}", flush=True)
        if self.adjoint:
            work = torch.empty(6 * nx * ny * nz, device="cuda")
            R.check(lib.rsg_e3d_backward_velocity_ws(C.byref(g), C.byref(s), work.data_ptr(), st), "velocity")
            R.check(lib.rsg_e3d_backward_stress(C.byref(g), C.byref(s), st), "stress")
        else:
            R.check(lib.rsg_e3d_forward_velocity(C.byref(g), C.byref(s), st), "velocity")
            R.check(lib.rsg_e3d_forward_stress(C.byref(g), C.byref(s), st), "stress")
        return [dev[k].cpu().numpy() for k in self.fields] + [t.cpu().numpy() for t in strips]

    def expect(self):
        if self.adjoint:
            self.o.velocity_bw()
            self.o.stress_bw()
        else:
            self.o.velocity()
            self.o.stress()
        return [getattr(self.o, k) for k in self.fields] + self.o.strips


@pytest.mark.parametrize("size", SIZES + INNER, ids=str)
def test_a3d_half_steps(size):
    s = _A3D(size)
    for name, got, want in zip(s.names, s.step(), s.expect()):
        _compare(name, got, want)


@pytest.mark.parametrize("adjoint", [False, True], ids=["forward", "adjoint"])
@pytest.mark.parametrize("size", SIZES + INNER + SHORT, ids=str)
def test_e3d_half_steps(size, adjoint):
    s = _E3D(size, adjoint)
    for name, got, want in zip(s.names, s.step(), s.expect()):
        _compare(name, got, want)


@pytest.mark.parametrize("kind", ["acoustic", "elastic", "elastic adjoint"])
def test_chunks_and_tile_orders_give_identical_fields(kind):
    """Every chunk length and both tile orders compute a cell alike: fields and
    strips bit for bit, on grids whose columns split over the XCDs unevenly."""
    from rockseis_amd import _lib as R
    old = R.get_tuning("zc3d"), R.get_tuning("xcd3d")
    try:
        for size in INNER + SIZES[2:4]:
            s = _A3D(size) if kind == "acoustic" else _E3D(size, kind.endswith("adjoint"))
            first = None
            for xcd in (1, 0):
                for zc in (0, 1, 3, 8, 16):
                    R.set_tuning("xcd3d", xcd)
                    R.set_tuning("zc3d", zc)
                    out = s.step()
                    first = first or out
                    for name, a, b in zip(s.names, out, first):
                        assert np.array_equal(a, b), (size, xcd, zc, name)
    finally:
        R.set_tuning("zc3d", old[0])
        R.set_tuning("xcd3d", old[1])
