"""The 2D tiles (rsg_fd2d.h) against the FP32 oracle on random states: one
modelling step with sources in the stress launch, and one step of the elastic
adjoint state, at the sizes where a boundary tile can go wrong (one tile with
both strips of an axis, one cell more and less than a tile, strips thinner
than the stencil, every stencil order), sources on tile corners sharing cells.

Moduli of about 1e4 make dt M / dx about one, and the wavelets are scaled to
source terms of about one: what a step adds is as large as the field it is added
to, so one cell of 10^4 off by 0.1% of the field, or a coefficient off by 2e-5,
shows.

Bound: an updated cell is a sum of up to 2 (2 order + 3) products and four
source terms; with |terms| about four times the result in the 2-norm of a
random state, two orders of summing them differ by at most 4 * 42 / 2 units of
2^-24, 5e-6."""
import ctypes as C

import numpy as np
import pytest

from tests.gpu_util import RTOL_L2, rel_l2

pytestmark = pytest.mark.gpu

# padded nx, nz, lpml, order
SIZES = [(64, 8, 1, 1), (65, 9, 2, 2), (40, 23, 6, 3), (160, 50, 18, 4), (127, 17, 4, 5), (129, 33, 9, 6), (18, 18, 5, 7),
         (63, 41, 3, 8), (200, 64, 20, 8), (200, 72, 12, 5)]
MODEL = {"a2d": ("L", "Rx", "Rz"), "e2d": ("L", "L2M", "M", "Rx", "Rz")}
FIELDS = {"a2d": ("P", "Vx", "Vz"), "e2d": ("Vx", "Vz", "Sxx", "Szz", "Sxz")}


@pytest.mark.parametrize("size", SIZES, ids=str)
@pytest.mark.parametrize("what", ["a2d", "e2d", "e2d adjoint"])
def test_steps(what, size):
    import torch
    from oracle import runs
    from rockseis_amd import _lib as R
    kind, adjoint = what[:3], "adjoint" in what
    nx, nz, lpml, order = size
    fs = int(kind == "e2d" and order % 2)
    rng = np.random.default_rng(sum(size))
    model = [rng.uniform(0.5e4, 1.5e4, (nz, nx)).astype(np.float32) for _ in MODEL[kind]]
    if kind == "a2d":
        o = runs.A2DState(*model, lpml, order, 10.0, 8.0, 1.5e-3)
    else:
        o = runs.E2DState(*model, lpml, order, 10.0, 8.0, 1.5e-3, fs)
    for a in [getattr(o, k) for k in FIELDS[kind]] + list(o.strips.values()):
        a[...] = rng.standard_normal(a.shape)
    cuda = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    dev = {k: cuda(getattr(o, k).copy()) for k in FIELDS[kind] + MODEL[kind] + ("tab",)}
    strips = {k: cuda(a.copy()) for k, a in o.strips.items()}
    g = R.Grid(nx=nx, ny=1, nz=nz, lpml=lpml, order=order, fs=fs, dx=10.0, dy=1.0, dz=8.0, dt=1.5e-3)
    s = R.State()
    for k, t in dev.items():
        setattr(s, k, t.data_ptr())
    for i, k in enumerate(R.A2D_STRIPS if kind == "a2d" else R.E2D_STRIPS):
        s.psi[i] = strips[k].data_ptr()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    lib = R.lib()
    print(f"{what} {size}", flush=True)
    if adjoint:
        R.check(lib.rsg_e2d_backward_velocity(C.byref(g), C.byref(s), st), "velocity")
        R.check(lib.rsg_e2d_backward_stress(C.byref(g), C.byref(s), st), "stress")
        o.velocity_bw()
        o.stress_bw()
    else:
        # the last cell before a tile edge, the first after it, the same cell
        # twice, and a trace outside the grid
        x, z = min(63, nx - 2) - lpml, min(7, nz - 2) - lpml
        x, z = max(x, 0), max(z, 0)
        smap = np.array([[x, z], [x, z], [max(x - 1, 0), z], [-1, 0]], np.int32)
        shift = rng.uniform(0, 1, (4, 2)).astype(np.float32)
        # acoustic: dt L w; elastic: dt w
        wav = ((0.1 if kind == "a2d" else 1e3) * rng.standard_normal((4, 1))).astype(np.float32)
        t = [cuda(a) for a in (smap, shift, wav)]
        src = R.Traces(R.PRESSURE, 4, 1, t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), None)
        code = R.KIND_A2D if kind == "a2d" else R.KIND_E2D
        # a chunk above 1 asks for the fused launches also for one step
        R.check(lib.rsg_modelling_run(code, C.byref(g), C.byref(s), C.byref(src), 0, None, 0, 1, 2, st), "step")
        o.velocity()
        o.stress()
        for F, M in [(o.P, o.L)] if kind == "a2d" else [(o.Sxx, None), (o.Szz, None)]:
            runs.inject2d(F, M, lpml, 1.5e-3, smap, shift, wav, 0)
    for k in FIELDS[kind]:
        e = rel_l2(dev[k].cpu().numpy(), getattr(o, k))
        assert e <= RTOL_L2, f"{k}: rel L2 {e:.2e}"
    for k, a in o.strips.items():
        e = rel_l2(strips[k].cpu().numpy(), a)
        assert e <= RTOL_L2, f"{k}: rel L2 {e:.2e}"
