"""The workloads whose speed is tracked: modelling runs, FWI gradients and RTM
images through the package's class API, over the sizes, orders, storage kinds
and adjoints it is used with.

listed() names them, draw(rng) makes more of the same ranges, prepare(case,
seed) builds what a program holds before the call (model, traces, plan),
run(state) makes one call, work(case) counts the memory traffic and arithmetic
the two-pass leapfrog cannot do without, tolerance(case) and exact(case, seed)
say what a result may differ by and what it is in 64 bits.
"""
import math

import numpy as np
import torch

from rockseis_amd import core, fwi, rtm

DER = [[1.0029], [1.188401, -7.046382e-2], [1.216624, -9.197724e-2, 1.300041e-2],
       [1.230862, -1.034123e-1, 2.011671e-2, -3.245760e-3],
       [1.239407, -1.105315e-1, 2.496329e-2, -5.804879e-3, 9.358680e-4],
       [1.245095, -1.153979e-1, 2.848442e-2, -7.899473e-3, 1.898222e-3, -2.935304e-4],
       [1.249150, -1.189375e-1, 3.116091e-2, -9.623004e-3, 2.812069e-3, -6.655106e-4, 9.728191e-5],
       [1.252186, -1.216289e-1, 3.326513e-2, -1.105777e-2, 3.647865e-3, -1.066144e-3, 2.437491e-4, -3.351959e-5]]


def _case(name, what, nx, nz, lpml, order, nt, ny=0, fs=False, src="P", shots=1, ncheck=0, store="fp32",
          adjoint="reference", mode="revolve", nhx=1, rec="P"):
    c = dict(what=what, nx=nx, nz=nz, lpml=lpml, order=order, nt=nt, ny=ny, fs=fs, src=src, shots=shots, ncheck=ncheck,
             store=store, adjoint=adjoint, mode=mode, nhx=nhx, rec=rec)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a small acoustic model, as in tests and first trials: every step is a few microseconds, launches count
        _case("a2d_mod_small", "a2d_mod", 121, 97, 20, 4, 300),
        # the plain acoustic 2D modelling workload (401 x 401, order 4), half its length
        _case("a2d_mod", "a2d_mod", 401, 401, 30, 4, 1000),
        # the elastic 2D modelling workload of the benchmark (2001 x 1001, order 8, vx and vz records), fewer steps
        _case("e2d_mod", "e2d_mod", 2001, 1001, 40, 8, 200, rec="VXVZ"),
        # an odd-sized elastic model with a free surface, a vertical force and pressure records
        _case("e2d_mod_odd", "e2d_mod", 1203, 517, 25, 6, 300, fs=True, src="VZ", rec="P"),
        # one shot of acoustic 3D modelling on a grid well beyond the caches
        _case("a3d_mod", "a3d_mod", 280, 240, 20, 4, 60, ny=260),
        # one shot of elastic 3D modelling with a free surface
        _case("e3d_mod", "e3d_mod", 160, 140, 20, 8, 50, ny=150, fs=True, rec="VZ"),
        # the batched acoustic 2D gradient on the benchmark's grid: Revolve, FP32 checkpoints
        _case("a2d_fwi", "a2d_fwi", 801, 401, 30, 8, 160, shots=8, ncheck=20),
        # elastic 2D gradients of uneven aperture windows on a persistent plan, 16-bit checkpoints
        _case("e2d_fwi", "e2d_fwi", 1600, 400, 30, 8, 120, shots=6, ncheck=12, store="s16"),
        # acoustic 3D gradient of one shot, 16-bit checkpoints
        _case("a3d_fwi", "a3d_fwi", 120, 100, 20, 4, 100, ny=110, ncheck=12, store="s16"),
        # the exact discrete adjoint in 3D (gradient checks, line searches that need it)
        _case("a3d_fwi_exact", "a3d_fwi", 90, 70, 15, 4, 60, ny=80, ncheck=10, adjoint="exact"),
        # elastic 3D gradient of one shot with a free surface
        _case("e3d_fwi", "e3d_fwi", 100, 80, 20, 8, 80, ny=90, fs=True, ncheck=12, store="s16"),
        # reverse-time migration of a batch of shots with subsurface offsets
        _case("a2d_rtm", "a2d_rtm", 601, 301, 30, 8, 200, shots=8, ncheck=20, nhx=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, its sizes spread over their logarithms, and the
    step count cut so that it costs no more than the listed case of its kind."""
    what = rng.choice(["a2d_mod", "e2d_mod", "a3d_mod", "e3d_mod", "a2d_fwi", "e2d_fwi", "a3d_fwi", "e3d_fwi", "a2d_rtm"])
    order = rng.choice([2, 4, 6, 8])
    lpml = rng.randint(10, 40)
    if what in ("a2d_mod", "e2d_mod"):
        c = _case(None, what, _log(rng, 90, 2000), _log(rng, 80, 1000), lpml, order, rng.randint(80, 400),
                  fs=rng.random() < 0.4, src="P" if what == "a2d_mod" else rng.choice(["P", "P", "VX", "VZ"]),
                  rec="P" if what == "a2d_mod" else rng.choice(["P", "VXVZ"]))
        cap = 2e8 if what == "a2d_mod" else 4e8
    elif what in ("a3d_mod", "e3d_mod"):
        top = 280 if what == "a3d_mod" else 160
        c = _case(None, what, _log(rng, 40, top), _log(rng, 40, top), rng.randint(8, 20), order, rng.randint(30, 90),
                  ny=_log(rng, 40, top), fs=rng.random() < 0.4, src="P" if what == "a3d_mod" else rng.choice(["P", "VX", "VY", "VZ"]),
                  rec="P" if what == "a3d_mod" else rng.choice(["VX", "VY", "VZ"]))
        cap = 1.5e9 if what == "a3d_mod" else 3e8
    elif what in ("a2d_fwi", "a2d_rtm"):
        c = _case(None, what, _log(rng, 100, 800), _log(rng, 80, 400), lpml, order, rng.randint(60, 200),
                  fs=rng.random() < 0.4, shots=rng.randint(1, 8), ncheck=rng.randint(6, 30),
                  nhx=rng.choice([1, 3, 7]) if what == "a2d_rtm" else 1)
        if what == "a2d_fwi":
            c["mode"] = rng.choice(["revolve", "revolve", "store"])
            c["store"] = rng.choice(["fp32", "s16"])
        cap = 4e8
    elif what == "e2d_fwi":
        c = _case(None, what, _log(rng, 300, 1600), _log(rng, 80, 400), rng.randint(10, 30), order, rng.randint(60, 130),
                  fs=rng.random() < 0.4, src=rng.choice(["P", "VZ"]), shots=rng.randint(1, 6), ncheck=rng.randint(6, 20),
                  store=rng.choice(["fp32", "s16"]))
        cap = 2.5e8
    else:
        top = 120 if what == "a3d_fwi" else 100
        c = _case(None, what, _log(rng, 30, top), _log(rng, 30, top), rng.randint(8, 20), order, rng.randint(30, 80),
                  ny=_log(rng, 30, top), fs=rng.random() < 0.4, ncheck=rng.randint(6, 20), store=rng.choice(["fp32", "s16"]))
        if what == "a3d_fwi" and rng.random() < 0.3:
            c.update(adjoint="exact", store="fp32")
            c["nx"], c["ny"], c["nz"] = min(c["nx"], 90), min(c["ny"], 80), min(c["nz"], 70)
            c["lpml"], c["nt"] = min(c["lpml"], 15), min(c["nt"], 60)
        cap = 3e8 if what == "a3d_fwi" else 1.6e8
    cells = _cells(c) * c["shots"]
    c["nt"] = max(20, min(c["nt"], int(cap / cells)))
    c["ncheck"] = min(c["ncheck"], c["nt"] // 2)
    return c


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _step(c):
    return 10.0 if c["what"] != "e2d_mod" else 5.0


def _dt(c):
    """80% of the stability bound the drivers check, for the fastest model."""
    n = 3 if c["ny"] else 2
    return float(np.float32(0.8 * 2.0 / (3.1415 * math.sqrt(n) / _step(c) * 4500.0)))


def _ricker(nt, dt, f0, t0):
    a = (np.pi * f0 * (np.arange(nt) * dt - t0)) ** 2
    return ((1.0 - 2.0 * a) * np.exp(-a)).astype(np.float32)


def _model(c, gen):
    """Vp: a linear gradient in depth times smooth anomalies of up to 10%; Vs = Vp / 1.8; Gardner's density."""
    shape = (c["nz"], c["ny"], c["nx"]) if c["ny"] else (c["nz"], c["nx"])
    coarse = torch.rand([1, 1] + [max(3, n // 25) for n in shape], generator=gen, device="cuda") * 0.2 - 0.1
    an = torch.nn.functional.interpolate(coarse, size=shape, mode="trilinear" if c["ny"] else "bilinear", align_corners=True)
    z = torch.linspace(0, 1, c["nz"], device="cuda").reshape([-1] + [1] * (len(shape) - 1))
    vp = ((1500.0 + 2400.0 * z) * (1.0 + an[0, 0])).float()
    return [a.cpu().numpy() for a in (vp, vp / 1.8, 0.31 * vp ** 0.25)]


def _inputs(c, seed):
    """Everything of a case that its seed decides, as numpy arrays."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    rng = np.random.RandomState(int(seed) % (1 << 31))
    wrng = np.random.RandomState(c["nx"] * 7 + c["nz"])  # the windows belong to the survey, not to its data
    d, dt, nt = _step(c), _dt(c), c["nt"]
    vp, vs, rho = _model(c, gen)
    f0 = 0.5 * 1500.0 / (5.0 * d)  # ten points a wavelength at the slowest cell
    t0 = min(1.0 / f0, 0.35 * nt * dt)
    if c["ny"]:
        gx, gy = np.meshgrid(np.arange(2, c["nx"] - 2, max(1, c["nx"] // 40)), np.arange(2, c["ny"] - 2, max(1, c["ny"] // 40)))
        g = np.stack([gx.ravel() * d, gy.ravel() * d, np.full(gx.size, 2.25 * d)], 1).astype(np.float32)
    else:
        g = np.stack([np.arange(2, c["nx"] - 2) * d, np.full(c["nx"] - 4, 2.25 * d)], 1).astype(np.float32)
    shots = []
    for k in range(c["shots"]):
        # aperture windows of a ragged batch are cut from the one model; elsewhere a shot sees all of it
        x0, nxw = 0, c["nx"]
        if c["what"] == "e2d_fwi":
            nxw = int(wrng.randint(max(60, c["nx"] * 3 // 8), max(61, c["nx"] * 5 // 8) + 1))
            x0 = int(wrng.randint(0, c["nx"] - nxw + 1))
        sx = x0 + int(rng.randint(nxw // 4, 3 * nxw // 4)) + 0.25
        s = [sx * d, 2.5 * d]
        if c["ny"]:
            s.insert(1, (rng.randint(c["ny"] // 4, 3 * c["ny"] // 4) + 0.5) * d)
        gk = g[x0:x0 + nxw - 4] if not c["ny"] else g
        wav = (_ricker(nt, dt, f0, t0) * rng.uniform(0.7, 1.3)).astype(np.float32)[None]
        # observed data: a direct and a reflected arrival with moveout
        r = np.linalg.norm(gk - np.float32([s]), axis=1)[:, None]
        obs = 0.0
        for t1, a in ((r / 1550.0, 1.0), (np.sqrt(r * r + (30 * d) ** 2) / 1900.0, 0.5)):
            q = (np.pi * f0 * (np.arange(nt)[None] * dt - t0 - t1)) ** 2
            obs = obs + a / (1.0 + r / (10 * d)) * (1 - 2 * q) * np.exp(-q)
        shots.append(dict(s=np.float32([s]), wav=wav, g=gk, x0=x0, nxw=nxw, obs=obs.astype(np.float32)))
    return dict(vp=vp, vs=vs, rho=rho, shots=shots, d=d, dt=dt)


# amplitude of the observed data against the modelled one: pressure in acoustic
# runs, and in elastic ones the records' own size
AMP = dict(a2d_fwi=200.0, a2d_rtm=200.0, a3d_fwi=100.0, e2d_fwi=1e-4, e3d_fwi=1e-5)
AMPV = dict(e2d_fwi=2e-8, e3d_fwi=1e-9)


def _traces(dim, coords, nt, dt, field, model, maptype, data=None):
    t = (core.Data3D if dim == 3 else core.Data2D)(coords.shape[0], nt, dt, 0.0, field)
    (t.scoords if maptype == core.SMAP else t.gcoords)[:] = coords
    if data is not None:
        t.data[:] = data
    t.makeMap(model, maptype)
    return t


def prepare(case, seed):
    c, i = case, _inputs(case, seed)
    d, dt, nt, what = i["d"], i["dt"], c["nt"], c["what"]
    sh = i["shots"][0]
    if what in ("a2d_fwi", "a2d_rtm"):
        shots = [fwi.Shot(s["s"], s["wav"], s["g"], s["obs"] * AMP[what]) for s in i["shots"]]
        sv = fwi.Survey(shots, c["lpml"], d, d, dt, order=c["order"], fs=c["fs"], ncheck=c["ncheck"], mode=c["mode"], fp16=c["store"])
        if what == "a2d_rtm":
            return dict(c=c, sv=sv, m=(i["vp"], i["rho"]))
        return dict(c=c, sv=sv, m=[torch.from_numpy(i[n]).cuda() for n in ("vp", "rho")])
    if what == "e2d_fwi":
        shots = [fwi.ElasticShot(s["s"], s["wav"], s["g"], np.stack([s["obs"] * AMP[what], s["obs"] * AMPV[what], s["obs"] * AMPV[what]]),
                                 s["x0"], s["nxw"], c["src"]) for s in i["shots"]]
        sv = fwi.ElasticSurvey(shots, c["lpml"], d, d, dt, order=c["order"], fs=c["fs"], ncheck=c["ncheck"], fp16=c["store"])
        m = [torch.from_numpy(i[n]).cuda() for n in ("vp", "vs", "rho")]
        return dict(c=c, m=m, plan=fwi.ElasticFwiPlan(*m, sv, tune=False))
    dim, elastic = 3 if c["ny"] else 2, what[0] == "e"
    cls = {"a2": core.ModelAcoustic2D, "e2": core.ModelElastic2D, "a3": core.ModelAcoustic3D, "e3": core.ModelElastic3D}[what[:2]]
    size = (c["nx"], c["ny"], c["nz"]) if dim == 3 else (c["nx"], c["nz"])
    m = cls(*size, c["lpml"], *([d] * dim), *([0.0] * dim), c["fs"])
    m.Vp[:], m.R[:] = i["vp"], i["rho"]
    if elastic:
        m.Vs[:] = i["vs"]
    m.staggerModels()
    src = _traces(dim, sh["s"], nt, dt, c["src"], m, core.SMAP, sh["wav"])
    st = dict(c=c, m=m, src=src)
    if what.endswith("_mod"):
        fields = ["VX", "VZ"] if c["rec"] == "VXVZ" else [c["rec"]]
        st["recs"] = {f: _traces(dim, sh["g"], nt, dt, f, m, core.GMAP) for f in fields}
    elif what == "a3d_fwi":
        st["obs"] = [_traces(3, sh["g"], nt, dt, "P", m, core.GMAP, sh["obs"] * AMP[what])]
    else:
        st["obs"] = [_traces(3, sh["g"], nt, dt, f, m, core.GMAP, sh["obs"] * AMPV[what]) for f in ("VX", "VY", "VZ")]
    return st


_MOD = dict(a2d_mod=core.ModellingAcoustic2D, e2d_mod=core.ModellingElastic2D, a3d_mod=core.ModellingAcoustic3D,
            e3d_mod=core.ModellingElastic3D)
_STATE = dict(a2d_mod=("P", "Vx", "Vz"), e2d_mod=("Sxx", "Szz", "Sxz", "Vx", "Vz"), a3d_mod=("P", "Vx", "Vy", "Vz"),
              e3d_mod=("Vx", "Vy", "Vz", "Sxx", "Syy", "Szz", "Syz", "Sxz", "Sxy"))


def run(state):
    c = state["c"]
    what = c["what"]
    if what.endswith("_mod"):
        mod = _MOD[what](state["m"], state["src"], c["order"], 1)
        for f, r in state["recs"].items():
            getattr(mod, {"P": "setRecP", "VX": "setRecVx", "VY": "setRecVy", "VZ": "setRecVz"}[f])(r)
        mod.run()
        out = {f: getattr(mod.waves, f) for f in _STATE[what]}
        out.update({"rec" + f: r.data for f, r in state["recs"].items()})
        return out
    if what == "a2d_fwi":
        mis, gv, gr, dmod = fwi.batch_gradient(*state["m"], state["sv"])
        return dict(misfit=mis, vp=gv, rho=gr, dmod=dmod)
    if what == "a2d_rtm":
        return dict(image=rtm.batch_image(*state["m"], state["sv"], nhx=c["nhx"]))
    if what == "e2d_fwi":
        state["plan"].set_model(*state["m"])
        mis, gvp, gvs, gr, outs = state["plan"].run()
        return dict(misfit=mis, vp=gvp, vs=gvs, rho=gr, dmod=[o["dmod"] for o in outs])
    m, obs = state["m"], state["obs"]
    if what == "a3d_fwi":
        f = fwi.FwiAcoustic3D(m, state["src"], obs[0], c["order"], 1)
        f.setAdjoint(c["adjoint"])
        img = dict(vp=fwi.Image3D(m), rho=fwi.Image3D(m))
        mod = [core.Data3D(obs[0].ntrace, c["nt"], obs[0].dt)]
        f.setDatamodP(mod[0])
    else:
        f = fwi.FwiElastic3D(m, state["src"], *obs, c["order"], 1)
        img = dict(vp=fwi.Image3D(m), vs=fwi.Image3D(m), rho=fwi.Image3D(m))
        mod = [core.Data3D(o.ntrace, c["nt"], o.dt) for o in obs]
        f.setDatamodUx(mod[0])
        f.setDatamodUy(mod[1])
        f.setDatamodUz(mod[2])
        f.setVsgrad(img["vs"])
    f.setVpgrad(img["vp"])
    f.setRhograd(img["rho"])
    f.setNcheck(c["ncheck"])
    f.setFp16Storage(c["store"])
    f.run_optimal()
    out = {n: v.imagedata for n, v in img.items()}
    out.update(misfit=float(f.misfit64), dmod=[t.data for t in mod])
    return out


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------

def _cells(c):
    L = c["lpml"]
    nx = c["nx"] / 2 if c["what"] == "e2d_fwi" else c["nx"]  # windows are half the model on average
    return (nx + 2 * L) * (c["nz"] + 2 * L) * ((c["ny"] + 2 * L) if c["ny"] else 1)


def _numforw(nt, snaps):
    """Forward steps of the binomial (Revolve) schedule."""
    reps, span = 0, 1
    while span < nt:
        reps += 1
        span = span * (reps + snaps) // reps
    return reps * nt - span * reps // (snaps + 1)


def work(case):
    """The two-pass leapfrog with every array of a half step read once and
    written once (4 bytes each: acoustic 2D 12, elastic 2D 20, acoustic 3D 16,
    elastic 3D 35 arrays a step), the steps of the checkpointing schedule, and
    for each reverse step the imaging condition's reads and updates."""
    c, what = case, case["what"]
    n, nt = _cells(c) * c["shots"], c["nt"]
    kind = what[:3]
    arrays = dict(a2d=12, e2d=20, a3d=16, e3d=35)[kind]
    nder = dict(a2d=4, e2d=8, a3d=6, e3d=18)[kind]
    if what.endswith("_mod"):
        fwd, rev, img = nt, 0, 0
    else:
        stored = c["mode"] == "store" and what == "a2d_fwi"
        fwd = nt if stored else _numforw(nt, c["ncheck"]) + 1
        rev = nt
        img = dict(a2d_fwi=3, a2d_rtm=2, e2d_fwi=12, a3d_fwi=7, e3d_fwi=21)[what]  # fields read; the images are shared
        if what in ("a3d_fwi", "e3d_fwi", "e2d_fwi"):
            img += 2 * (2 if what == "a3d_fwi" else 3)
        if c["adjoint"] == "exact":
            img = 8  # the forward half step and the four model-gradient sums
    return {"bytes": 4.0 * n * ((fwd + rev) * arrays + rev * img),
            "flops": n * ((fwd + rev) * (nder * (3.0 * c["order"] + 2)) + rev * 4.0 * img)}


def tolerance(case):
    """Relative 2-norm errors of about four times what the float32 path shows
    against 64 bits: wavefields after up to 1000 steps, gradients with FP32
    checkpoints, and gradients with 16-bit ones."""
    if case["what"] == "a2d_mod":
        return {"rel": 2.4e-5}
    if case["what"].endswith("_mod"):
        return {"rel": 6e-6}
    return {"rel": 1e-4 if case["store"] == "s16" else 1e-5}


# --------------------------------------------------------------------------
# The same in 64 bits, as plain torch
# --------------------------------------------------------------------------

def _profile(L, n, dt, stag):
    """A, B, C of the CFS-PML along one axis (zero between the layers)."""
    i = np.arange(L, dtype=np.float64)
    h = 0.5 if stag else 0.0
    tab = np.zeros((3, n))
    for side, func in ((slice(0, L), ((L - i - h) / L) ** 3), (slice(n - L, n), ((i + 1 + h) / L) ** 3)):
        k = 1.0 + func
        b = np.exp(-1200.0 * func / k * dt)
        tab[:, side] = (1.0 - b) / k, b, 1.0 - 1.0 / k
    return torch.from_numpy(tab).cuda()


class _Sim:
    """Velocity-stress stepping of one model in float64: P (acoustic) or the
    stresses S[a, b], and V[a], axes 0 = x, 1 = y or z, 2 = z, on the padded
    grid [.., z, (y), x]; derivatives as banded matrices with the reduced
    orders at the array's ends."""

    def __init__(self, c, m, d, dt, elastic, nb=1):
        self.dt, self.L, self.fs, self.elastic = dt, c["lpml"], c["fs"], elastic
        self.dim = 3 if c["ny"] else 2
        self.ax = range(self.dim)
        pad = lambda a: torch.nn.functional.pad(a[None, None], [self.L] * (2 * self.dim), mode="replicate")[0, 0]
        vp, rho = pad(m["vp"]), pad(m["rho"])
        self.shape = vp.shape
        n = [self.shape[self.dim - 1 - a] for a in self.ax]
        row = torch.zeros(n[-1], dtype=torch.float64, device="cuda")
        row[self.L] = 1.0 if c["fs"] else 0.0
        row = row.reshape([-1] + [1] * (self.dim - 1))  # the free-surface plane
        self.row = row

        def stag(a, axis):
            k = self.dim - 1 - axis
            s = (a.narrow(k, 0, a.shape[k] - 1) + a.narrow(k, 1, a.shape[k] - 1)) / 2
            return torch.cat([s, s.narrow(k, s.shape[k] - 1, 1)], k)

        self.R = [(1.0 / stag(rho, a)) * (1.0 + (row if a < self.dim - 1 else 0.0)) for a in self.ax]
        lam2mu = rho * vp * vp
        if elastic:
            vs = pad(m["vs"])
            mu = rho * vs * vs
            self.lam = (lam2mu - 2 * mu) * (1 - row)
            self.l2m = lam2mu * (1 - row) + mu * row
            self.mu = {(a, b): stag(stag(mu, a), b) for a in self.ax for b in self.ax if a < b}
        else:
            self.lam = lam2mu * (1 - row)
        self.prof = [[_profile(self.L, n[a], dt, s).reshape([3] + [-1 if k == self.dim - 1 - a else 1 for k in range(self.dim)])
                      for s in (0, 1)] for a in self.ax]
        self.D = [[self._matrix(n[a], c["order"], d, f) for f in (False, True)] for a in self.ax]
        self.nb = nb
        self.reset()

    def reset(self):
        z = torch.zeros((self.nb,) + tuple(self.shape), dtype=torch.float64, device="cuda")
        self.psi, self.V = {}, [z for _ in self.ax]
        self.P = z
        self.S = {(a, b): z for a in self.ax for b in self.ax if a <= b}

    @staticmethod
    def _matrix(n, order, d, fwd):
        m = np.zeros((n, n))
        for i in range(n):
            k = min(order, i + 1, n - 1 - i) if fwd else min(order, i, n - i)
            for j in range(k):
                lo, hi = (i - j, i + j + 1) if fwd else (i - j - 1, i + j)
                m[i, hi] += DER[k - 1][j] / d
                m[i, lo] -= DER[k - 1][j] / d
        return torch.from_numpy(m).cuda()

    def diff(self, key, f, a, fwd):
        """One derivative term with its memory variable's correction."""
        D = self.D[a][fwd]
        if a == 0:
            g = f @ D.T
        elif a == self.dim - 1:
            g = (D @ f.reshape(f.shape[0], f.shape[1], -1)).reshape(f.shape)
        else:
            g = D @ f
        A, B, C = self.prof[a][int(fwd)]
        p = A * g if key not in self.psi else B * self.psi[key] + A * g
        self.psi[key] = p
        return g - (p + C * g)

    def velocity(self, S=None):
        if not self.elastic:
            self.V = [v + self.dt * self.R[a] * self.diff(("p", a), self.P, a, True) for a, v in enumerate(self.V)]
            return
        S, new = S or self.S, []
        for a in self.ax:
            t = sum(self.diff(("s", a, b), S[min(a, b), max(a, b)], b, a == b) for b in self.ax)
            new.append(self.V[a] + self.dt * self.R[a] * t)
        self.V = new

    def stress(self, unit=False):
        if not self.elastic:
            self.P = self.P + self.dt * self.lam * sum(self.diff(("v", a), self.V[a], a, False) for a in self.ax)
            return
        e = [self.diff(("v", a, a), self.V[a], a, False) for a in self.ax]
        for a in self.ax:
            t = e[a] if unit else self.l2m * e[a] + self.lam * sum(e[b] for b in self.ax if b != a)
            s = self.S[a, a] + self.dt * t
            self.S[a, a] = s * (1 - self.row) if a == self.dim - 1 else s
            for b in self.ax:
                if a < b:
                    t = self.diff(("v", b, a), self.V[b], a, True) + self.diff(("v", a, b), self.V[a], b, True)
                    self.S[a, b] = self.S[a, b] + self.dt * (t if unit else self.mu[a, b] * t)

    def step(self):
        self.velocity()
        self.stress()

    def step_adjoint(self):
        """The elastic adjoint-state step: moduli-weighted stresses, unit moduli."""
        tot = sum(self.S[b, b] for b in self.ax)
        self.velocity({k: self.l2m * s + self.lam * (tot - s) if k[0] == k[1] else self.mu[k] * s for k, s in self.S.items()})
        self.stress(unit=True)

    def copy(self):
        return ([v for v in self.V], self.P, dict(self.S))


class _Points:
    """Trace positions of one field: flat cells of the batched grid and their
    multilinear weights, [shot, trace, corner]."""

    def __init__(self, sim, coords, orig, size, d, field):
        h = [-0.5 if field == "V" + "XYZ"[a if sim.dim == 3 or a == 0 else 2] else 0.0 for a in sim.ax]
        idx, wts = [], []
        n = [sim.shape[sim.dim - 1 - a] for a in sim.ax]
        for k, (cs, o) in enumerate(zip(coords, orig)):
            r = (cs.astype(np.float64) - np.asarray(o)) / d + np.asarray(h)
            p = np.floor(r).astype(np.int64)
            ok = ((p >= 0) & (p < np.asarray(size))).all(1)
            f = r - p
            ci, cw = [], []
            for corner in range(1 << sim.dim):
                at, w = np.int64(0), ok.astype(np.float64)
                for a in reversed(sim.ax):
                    b = (corner >> a) & 1
                    at = at * n[a] + np.clip(p[:, a], 0, None) + b + sim.L
                    w = w * (f[:, a] if b else 1.0 - f[:, a])
                ci.append(at)
                cw.append(w)
            idx.append(np.stack(ci, 1) + k * int(np.prod(n)))
            wts.append(np.stack(cw, 1))
        self.i, self.w = torch.from_numpy(np.stack(idx)).cuda(), torch.from_numpy(np.stack(wts)).cuda()

    def get(self, f):
        return (f.reshape(-1)[self.i] * self.w).sum(-1)

    def add(self, f, scale, val):
        """f plus scale (None: 1, or a field) times val[shot, trace] over the corners."""
        v = val[..., None] * self.w
        if scale is not None:
            v = v * scale.expand(f.shape).reshape(-1)[self.i]
        return f.reshape(-1).index_add(0, self.i.reshape(-1), v.reshape(-1)).reshape(f.shape)


def _source(sim, pts, field, w):
    if not sim.elastic:
        sim.P = pts.add(sim.P, sim.lam, sim.dt * w)
    elif field == "P":
        for a in sim.ax:
            sim.S[a, a] = pts.add(sim.S[a, a], None, -sim.dt * w)
    else:
        a = {"VX": 0, "VY": 1, "VZ": sim.dim - 1}[field]
        sim.V[a] = pts.add(sim.V[a], sim.R[a], sim.dt * w)


def _gather(sim, pts, field):
    if field == "P":
        return pts.get(sim.P) if not sim.elastic else pts.get(sum(sim.S[a, a] for a in sim.ax)) * 0.5
    return pts.get(sim.V[{"VX": 0, "VY": 1, "VZ": sim.dim - 1}[field]])


def _interior(f, sim, size, lo, hi, off=(0, 0, 0)):
    """The model's cells lo <= i < n - hi of every axis of a padded field, shifted by off."""
    for a in sim.ax:
        k = f.dim() - 1 - a
        f = f.narrow(k, sim.L + lo + off[a], size[a] - lo - hi)
    return f


def exact(case, seed):
    c, what = case, case["what"]
    i = _inputs(c, seed)
    d, dt, nt = float(np.float32(i["d"])), i["dt"], c["nt"]
    if what == "e2d_fwi":
        return _exact_windows(c, i, d, dt)
    m = {n: torch.from_numpy(i[n]).cuda().double() for n in ("vp", "vs", "rho")}
    if c["adjoint"] == "exact":
        for n in ("vp", "rho"):
            m[n].requires_grad_(True)
    elastic = what[0] == "e"
    sim = _Sim(c, m, d, dt, elastic, c["shots"])
    size = [c["nx"], c["ny"], c["nz"]] if c["ny"] else [c["nx"], c["nz"]]
    zero = [[0.0] * sim.dim] * c["shots"]
    at = lambda key, field: _Points(sim, [s[key] for s in i["shots"]], zero, size, d, field)
    wav = torch.from_numpy(np.stack([s["wav"] for s in i["shots"]])).cuda().double()
    src = at("s", c["src"])
    fields = ["VX", "VZ"] if c["rec"] == "VXVZ" else [c["rec"]]
    if what == "e3d_fwi":
        fields = ["VX", "VY", "VZ"]
    recs = {f: at("g", f) for f in fields}
    data, hist = {f: [] for f in fields}, []
    for t in range(nt):
        if not what.endswith("_mod") and c["adjoint"] != "exact":
            hist.append(sim.copy() if elastic else sim.P)
        sim.step()
        _source(sim, src, c["src"], wav[..., t])
        for f in fields:
            data[f].append(_gather(sim, recs[f], f))
    data = {f: torch.stack(v, -1) for f, v in data.items()}
    if what.endswith("_mod"):
        names = dict(Vx=lambda: sim.V[0], Vy=lambda: sim.V[1], Vz=lambda: sim.V[-1], P=lambda: sim.P)
        z = sim.dim - 1
        for n, k in dict(Sxx=(0, 0), Syy=(1, 1), Szz=(z, z), Syz=(1, z), Sxz=(0, z), Sxy=(0, 1)).items():
            names[n] = lambda k=k: sim.S[k]
        out = {n: names[n]()[0] for n in _STATE[what]}
        out.update({"rec" + f: v[0] for f, v in data.items()})
        return out
    amp = AMPV.get(what, AMP[what])
    obs = torch.from_numpy(np.stack([s["obs"] * np.float32(amp) for s in i["shots"]])).cuda().double()
    if what == "a2d_rtm":
        return dict(image=_rtm(c, sim, recs["P"], obs, hist, size))
    res = {f: v - obs for f, v in data.items()}
    mis = 0.5 * sum((r * r).sum() for r in res.values())
    if c["adjoint"] == "exact":
        mis.backward()
        return dict(misfit=float(mis), vp=m["vp"].grad, rho=m["rho"].grad, dmod=[data["P"][0].detach()])
    last = sim.copy() if elastic else sim.P
    sim.reset()
    if elastic:
        g = _elastic3_gradient(c, sim, recs, res, hist, last, m, size, d)
        return dict(misfit=float(mis), vp=g[0], vs=g[1], rho=g[2], dmod=[data[f][0] for f in fields])
    vg, rg = (torch.zeros(m["vp"].shape, dtype=torch.float64, device="cuda") for _ in range(2))
    hi = 1 if sim.dim == 2 else 0
    inner = tuple(slice(1, n - hi) for n in vg.shape)
    for t in range(nt - 1, -1, -1):
        if t < nt - 1:
            sim.step()
        sim.P = recs["P"].add(sim.P, sim.lam, dt * res["P"][..., t])
        a, b = _acoustic_image(sim, last if t == nt - 1 else hist[t], m, size, d, hi, inner)
        vg[inner] += a
        rg[inner] += b
    dm = data["P"]
    return dict(misfit=float(mis), vp=vg, rho=rg, dmod=dm if sim.dim == 2 else [dm[0]])


def _unit(dim, *k):
    """The offset -1 along each axis of k."""
    return tuple(-1 if a in k else 0 for a in range(dim))


def _acoustic_image(sim, P, m, size, d, hi, inner):
    at = lambda f, off=(0, 0, 0): _interior(f, sim, size, 1, hi, off)
    ws, div, corr = at(P), 0.0, 0.0
    for a in sim.ax:
        back, fore = _unit(sim.dim, a), tuple(-o for o in _unit(sim.dim, a))
        div = div + (at(sim.V[a]) - at(sim.V[a], back)) / d
        # the reference's 3D imaging condition reads Vz one cell back in y with Rz one cell back in z
        vback = _unit(3, 1) if sim.dim == 3 and a == 2 else back
        corr = corr + 0.5 * at(sim.V[a]) * at(sim.R[a]) * (at(P, fore) - ws) / d
        corr = corr + 0.5 * at(sim.V[a], vback) * at(sim.R[a], back) * (ws - at(P, back)) / d
    return (2.0 / m["vp"][inner] * ws * div).sum(0), (1.0 / m["rho"][inner] * ws * div + corr).sum(0)


def _rtm(c, sim, rec, obs, hist, size):
    last, nh = sim.P, c["nhx"]
    sim.reset()
    img = torch.zeros((1, nh, c["nz"], c["nx"]), dtype=torch.float64, device="cuda")
    for t in range(c["nt"] - 1, -1, -1):
        if t < c["nt"] - 1:
            sim.step()
        sim.P = rec.add(sim.P, sim.lam, sim.dt * obs[..., t])
        ws = _interior(last if t == c["nt"] - 1 else hist[t], sim, size, 0, 0)
        wr = _interior(sim.P, sim, size, 0, 0)
        for k in range(nh):
            h = k - (nh - 1) // 2
            lo, n = abs(h), c["nx"] - 2 * abs(h)
            img[0, k, :, lo:lo + n] += (ws[..., lo - h:lo - h + n] * wr[..., lo + h:lo + h + n]).sum(0)
    return img


def _exact_windows(c, i, d, dt):
    """Elastic 2D gradients window by window, stacked."""
    grads = [torch.zeros((c["nz"], c["nx"]), dtype=torch.float64, device="cuda") for _ in range(3)]
    total, dmods, nt = 0.0, [], c["nt"]
    for s in i["shots"]:
        x0, n = s["x0"], s["nxw"]
        m = {k: torch.from_numpy(np.ascontiguousarray(i[k][:, x0:x0 + n])).cuda().double() for k in ("vp", "vs", "rho")}
        sim, size = _Sim(c, m, d, dt, True), [n, c["nz"]]
        pts = lambda key, f: _Points(sim, [s[key]], [[x0 * d, 0.0]], size, d, f)
        src, wav = pts("s", c["src"]), torch.from_numpy(s["wav"])[None].cuda().double()
        recs = {f: pts("g", f) for f in ("P", "VX", "VZ")}
        data, hist = {f: [] for f in recs}, []
        for t in range(nt):
            hist.append(sim.copy())
            sim.step()
            _source(sim, src, c["src"], wav[..., t])
            for f in recs:
                data[f].append(_gather(sim, recs[f], f))
        last = sim.copy()
        data = {f: torch.stack(v, -1) for f, v in data.items()}
        amp = dict(P=AMP["e2d_fwi"], VX=AMPV["e2d_fwi"], VZ=AMPV["e2d_fwi"])
        res = {f: v - torch.from_numpy(s["obs"] * np.float32(amp[f])).cuda().double() for f, v in data.items()}
        total += float(0.5 * sum((r * r).sum() for r in res.values()))
        dmods.append([data[f][0] for f in ("P", "VX", "VZ")])
        sim.reset()
        lam, mu, rk = (torch.zeros((c["nz"], n), dtype=torch.float64, device="cuda") for _ in range(3))
        inner = (slice(1, -1), slice(1, -1))
        for t in range(nt - 1, -1, -1):
            if t < nt - 1:
                sim.step_adjoint()
            for f in recs:
                _source(sim, recs[f], f, res[f][..., t])
            V, _, S = last if t == nt - 1 else hist[t]
            at = lambda f, x=0, z=0: _interior(f, sim, size, 1, 1, (x, z)).reshape(c["nz"] - 2, n - 2)
            ws, wz, sxx, szz, sxz = V[0], V[1], S[0, 0], S[1, 1], S[0, 1]
            rx, rz, rxx, rzz, rxz = sim.V[0], sim.V[1], sim.S[0, 0], sim.S[1, 1], sim.S[0, 1]
            ex, ez = (at(ws) - at(ws, -1)) / d, (at(wz) - at(wz, 0, -1)) / d
            lam[inner] -= (ex + ez) * (at(rxx) + at(rzz))
            f2 = 0.0
            for x in (-1, 0):
                for z in (-1, 0):
                    # shear strain at the corner (x, z) of the cell
                    g = (at(ws, x, z + 1) - at(ws, x, z)) / d + (at(wz, x + 1, z) - at(wz, x, z)) / d
                    f2 = f2 + g * at(rxz, x, z)
            mu[inner] += 2.0 * (ex * at(rzz) + ez * at(rxx)) - 0.25 * f2
            Rx, Rz = sim.R
            u = 0.0
            for x in (-1, 0):
                u = u + 0.5 * at(rx, x) * at(Rx, x) * ((at(sxx, x + 1) - at(sxx, x)) + (at(sxz, x) - at(sxz, x, -1))) / d
            for z in (-1, 0):
                u = u + 0.5 * at(rz, 0, z) * at(Rz, 0, z) * ((at(sxz, 0, z) - at(sxz, -1, z)) + (at(szz, 0, z + 1) - at(szz, 0, z))) / d
            rk[inner] -= u
        vp, vs, rho = m["vp"], m["vs"], m["rho"]
        sl = (slice(None), slice(x0, x0 + n))
        grads[0][sl] += 2 * rho * vp * lam
        grads[1][sl] += 2 * rho * vs * (mu - 2 * lam)
        grads[2][sl] += (vp * vp - 2 * vs * vs) * lam + vs * vs * mu + rk
    return dict(misfit=total, vp=grads[0], vs=grads[1], rho=grads[2], dmod=dmods)


def _elastic3_gradient(c, sim, recs, res, hist, last, m, size, d):
    shape = m["vp"].shape
    lam, mu, rk = (torch.zeros(shape, dtype=torch.float64, device="cuda") for _ in range(3))
    inner = (slice(1, -1),) * 3
    at = lambda f, x=0, y=0, z=0: _interior(f, sim, size, 1, 1, (x, y, z)).reshape([n - 2 for n in shape])
    nt = c["nt"]
    for t in range(nt - 1, -1, -1):
        if t < nt - 1:
            sim.step_adjoint()
        for f in recs:
            _source(sim, recs[f], f, res[f][..., t])
        V, _, S = last if t == nt - 1 else hist[t]
        back = [_unit(3, a) for a in range(3)]
        e = [(at(V[a]) - at(V[a], *back[a])) / d for a in range(3)]
        r = [at(sim.S[a, a]) for a in range(3)]
        lam[inner] -= sum(e) * sum(r)
        g = 0.0
        for a, b in ((0, 1), (0, 2), (1, 2)):
            s = 0.0
            for i in (-1, 0):
                for j in (-1, 0):
                    o = [0, 0, 0]
                    o[a], o[b] = i, j
                    oa, ob = list(o), list(o)
                    oa[a] += 1
                    ob[b] += 1
                    s = s + (at(V[b], *oa) - at(V[b], *o)) / d + (at(V[a], *ob) - at(V[a], *o)) / d
            g = g + 0.25 * s * at(sim.S[a, b])
        mu[inner] -= g + 2.0 * sum(e[a] * r[a] for a in range(3))
        u = 0.0
        for a in range(3):
            for k in (0, -1):
                o = [0, 0, 0]
                o[a] = k
                # the reference reads the receiver's Vz one cell back in y where Rz and the stresses are one back in z
                v = at(sim.V[a], 0, k, 0) if a == 2 else at(sim.V[a], *o)
                t2 = 0.0
                for b in range(3):
                    p = S[min(a, b), max(a, b)]
                    q = list(o)
                    if a == b:
                        q[a] += 1
                        t2 = t2 + at(p, *q) - at(p, *o)
                    else:
                        q[b] -= 1
                        t2 = t2 + at(p, *o) - at(p, *q)
                u = u + 0.5 * v * at(sim.R[a], *o) * t2 / d
        rk[inner] -= u
    vp, vs, rho = m["vp"], m["vs"], m["rho"]
    return 2 * rho * vp * lam, 2 * rho * vs * (mu - 2 * lam), vp * vp * lam + vs * vs * mu + rk
