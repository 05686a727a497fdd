"""The 3D z march (rsg_fd3d.h) against the FP32 oracle on random states: one
velocity and one stress half step (acoustic; elastic, and its adjoint state's)
at the sizes where a tile, a chunk or a
strip can go wrong (rows of 64 and of 32, one cell more and less, strips
thinner than the stencil, chunks of odd length), every stencil order.

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
# the elastic steps also take grids shorter than the stencil
SHORT = [(9, 7, 8, 2, 8), (20, 70, 5, 1, 4)]


def _random(rng, *arrays):
    for a in arrays:
        a[...] = rng.standard_normal(a.shape)


def _compare(name, got, want):
    e = rel_l2(got, want)
    assert e <= RTOL_L2, f"{name}: rel L2 {e:.2e}"


@pytest.mark.parametrize("size", SIZES, ids=str)
def test_a3d_half_steps(size):
    import torch
    from oracle import runs
    from rockseis_amd import _lib as R
    nx, ny, nz, lpml, order = size
    rng = np.random.default_rng(sum(size))
    model = [rng.uniform(0.5, 1.5, (nz, ny, nx)).astype(np.float32) for _ in range(4)]
    o = runs.A3DState(*model, lpml, order, 10.0, 12.5, 8.0, 1.5e-3)
    _random(rng, o.P, o.Vx, o.Vy, o.Vz, *o.strips.values())
    dev = {k: torch.from_numpy(getattr(o, k).copy()).cuda() for k in ("P", "Vx", "Vy", "Vz", "L", "Rx", "Ry", "Rz", "tab")}
    strips = {k: torch.from_numpy(a.copy()).cuda() for k, a in o.strips.items()}
    g = R.Grid(nx=nx, ny=ny, nz=nz, lpml=lpml, order=order, fs=0, dx=10.0, dy=12.5, dz=8.0, dt=1.5e-3)
    s = R.State()
    for k, t in dev.items():
        setattr(s, k, t.data_ptr())
    for i, k in enumerate(R.A3D_STRIPS):
        s.psi[i] = strips[k].data_ptr()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    print(f"a3d {size}", flush=True)
    R.check(R.lib().rsg_a3d_forward_velocity(C.byref(g), C.byref(s), st), "velocity")
    R.check(R.lib().rsg_a3d_forward_stress(C.byref(g), C.byref(s), st), "stress")
    o.velocity()
    o.stress()
    for k in ("P", "Vx", "Vy", "Vz"):
        _compare(k, dev[k].cpu().numpy(), getattr(o, k))
    for k, a in o.strips.items():
        _compare(k, strips[k].cpu().numpy(), a)


@pytest.mark.parametrize("adjoint", [False, True], ids=["forward", "adjoint"])
@pytest.mark.parametrize("size", SIZES + SHORT, ids=str)
def test_e3d_half_steps(size, adjoint):
    import torch
    from oracle import runs
    from rockseis_amd import _lib as R
    nx, ny, nz, lpml, order = size
    fs = order % 2
    rng = np.random.default_rng(sum(size))
    names = ("L", "L2M", "Mxz", "Myz", "Mxy", "Rx", "Ry", "Rz")
    o = runs.E3DState([rng.uniform(0.5, 1.5, (nz, ny, nx)) for _ in names], lpml, order, (10.0, 12.5, 8.0), 1.5e-3, fs)
    _random(rng, *(getattr(o, k) for k in runs.E3D_FIELDS), *o.strips)
    dev = {k: torch.from_numpy(getattr(o, k).copy()).cuda() for k in runs.E3D_FIELDS + names + ("tab",)}
    strips = [torch.from_numpy(a.copy()).cuda() for a in o.strips]
    g = R.Grid(nx=nx, ny=ny, nz=nz, lpml=lpml, order=order, fs=fs, dx=10.0, dy=12.5, dz=8.0, dt=1.5e-3)
    s = R.StateE3D()
    for k, t in dev.items():
        setattr(s, k, t.data_ptr())
    for i, t in enumerate(strips):
        s.psi[i] = t.data_ptr()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    lib = R.lib()
    print(f"e3d {size} adjoint {adjoint}", flush=True)
    if adjoint:
        work = torch.empty(6 * nx * ny * nz, device="cuda")
        R.check(lib.rsg_e3d_backward_velocity_ws(C.byref(g), C.byref(s), work.data_ptr(), st), "velocity")
        R.check(lib.rsg_e3d_backward_stress(C.byref(g), C.byref(s), st), "stress")
        o.velocity_bw()
        o.stress_bw()
    else:
        R.check(lib.rsg_e3d_forward_velocity(C.byref(g), C.byref(s), st), "velocity")
        R.check(lib.rsg_e3d_forward_stress(C.byref(g), C.byref(s), st), "stress")
        o.velocity()
        o.stress()
    for k in runs.E3D_FIELDS:
        _compare(k, dev[k].cpu().numpy(), getattr(o, k))
    for i, a in enumerate(o.strips):
        _compare(f"strip {i}", strips[i].cpu().numpy(), a)
