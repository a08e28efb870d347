"""The work that is timed: what a host model has this library do, through
``efdc_amd.lib.Context`` and ``efdc_amd.adjoint.DyeMisfit``.

A case is one of these kinds of pass:

``external``  one CALPUV2C step (assembly, CONGRAD, transports, depths) on an
              irregular lake or, with ``isdry``, on a drying tidal basin;
``hydro``     one hydrodynamic step, CALPUV2C then CALUVW (sigma layers), on a
              tidal basin;
``transport`` a segment of CALCONC steps of ``nconst`` constituents on a given
              flow, ending in a device snapshot (the model's checkpoint, and
              the way to the constituents without leaving the GPU);
``step``      a segment of whole steps (closure or CALUVW, CALPUV2C, CALCONC)
              of one tidal basin, ending in a device snapshot;
``ensemble``  the same for many basins held in one context;
``adjoint``   a gradient of the dye misfit: checkpointed forward run and
              reverse sweep;
``restart``   RESTART.OUT's text of the whole state, in host memory.

Outputs are the context's own device arrays, or views of the snapshot.
``exact`` restates the steps in plain torch, FP64.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("efdcplus8.5_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from efdc_amd import abi, adjoint, grids, lib  # noqa: E402

G = 9.81
PI2 = 2.0 * 3.1415926535898  # the model's own PI
NH, NK, NW = 64, 14, 2       # horizontal, layer and interface arrays of a snapshot

EXT_OUT = ("P", "HP", "UHDYE", "VHDXE", "UHE", "VHE", "HU", "HV", "HUI", "HVI", "HPI")
UVW_OUT_K = ("UHDYF", "VHDXF", "UHDY", "VHDX", "U", "V", "UHDYF2", "VHDXF2", "UHDYEK",
             "VHDXEK", "UHDY2", "VHDX2", "U2", "V2", "HPK", "HPKI")
STEP_OUT_K = ("HPK", "H1PK", "HPKI", "UHDY2", "VHDX2")
UVW_OUT_H = ("UHDYE", "VHDXE", "P", "HP", "HPI", "HU", "HV", "UHE", "VHE", "UV", "VU")


def listed():
    return [
        # a small calibration basin with every option of a tidal run, FP64
        # (the test and smoke sizes): latency and launches
        dict(name="step small fp64", kind="step", nx=128, ny=64, kc=5, store="fp64", cg="fp64",
             internal=0, steps=8),
        # the benchmark lake: the external solve at scale, FP32-refined
        dict(name="lake 1024 mixed", kind="external", nx=1024, ny=1024, cg="mixed", isdry=0),
        # an ordinary lake with odd sizes in the default FP64 solve
        dict(name="lake 417x291 fp64", kind="external", nx=417, ny=291, cg="fp64", isdry=0),
        # a lake that no longer fits one co-resident solve
        dict(name="lake 1800 mixed", kind="external", nx=1800, ny=1700, cg="mixed", isdry=0),
        # tidal flats, cells drying and wetting within the step
        dict(name="drying 600x400 fp64", kind="external", nx=600, ny=400, cg="fp64", isdry=99),
        # water quality on a given flow: FP32 storage, settling sediment
        dict(name="transport large fp32", kind="transport", nx=640, ny=512, kc=20, nconst=4,
             store="fp32", adac=0, steps=16),
        # the same in FP64 with anti-diffusion and the flux limiter, odd sizes
        dict(name="transport adac fp64", kind="transport", nx=253, ny=187, kc=9, nconst=3,
             store="fp64", adac=1, steps=8),
        # 3-D hydrodynamics
        dict(name="hydro 3-D large", kind="hydro", nx=640, ny=400, kc=20, store="fp32",
             cg="mixed"),
        # a 3-D run of ordinary size with its transport
        dict(name="step 3-D medium", kind="step", nx=211, ny=165, kc=10, store="fp32", cg="fp64",
             internal=1, steps=8),
        # a parameter study: many small basins at once
        dict(name="ensemble 40 basins", kind="ensemble", nb=40, kc=6, store="fp64", cg="fp64",
             steps=4),
        # a source inversion: the gradient of one window
        dict(name="adjoint gradient", kind="adjoint", nx=200, kc=8, nsrc=8, nobs=40, nsteps=20,
             every=5, ckpt=10, store="fp32"),
        # a restart file of a 3-D run
        dict(name="restart text", kind="restart", nx=96, ny=80, kc=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("external", "external", "drying", "transport", "transport", "adac",
                       "hydro", "step", "step", "ensemble", "adjoint", "restart"))
    if kind == "external":
        return dict(kind="external", nx=_log(rng, 40, 1600), ny=_log(rng, 40, 1600),
                    cg=rng.choice(("fp64", "mixed")), isdry=0)
    if kind == "drying":
        return dict(kind="external", nx=_log(rng, 48, 700), ny=_log(rng, 24, 450),
                    cg=rng.choice(("fp64", "mixed")), isdry=rng.choice((1, 99)))
    if kind == "transport":
        return dict(kind="transport", nx=_log(rng, 40, 640), ny=_log(rng, 40, 500),
                    kc=rng.randint(1, 20), nconst=rng.randint(1, 4),
                    store=rng.choice(("fp32", "fp64")), adac=0, steps=8)
    if kind == "adac":
        return dict(kind="transport", nx=_log(rng, 40, 250), ny=_log(rng, 40, 190),
                    kc=rng.randint(2, 9), nconst=rng.randint(1, 3),
                    store=rng.choice(("fp32", "fp64")), adac=1, steps=4)
    if kind == "hydro":
        return dict(kind="hydro", nx=_log(rng, 40, 500), ny=_log(rng, 30, 400),
                    kc=rng.randint(2, 20), store=rng.choice(("fp32", "fp64")),
                    cg=rng.choice(("fp64", "mixed")))
    if kind == "step":
        return dict(kind="step", nx=_log(rng, 32, 300), ny=_log(rng, 24, 200),
                    kc=rng.randint(1, 10), store=rng.choice(("fp32", "fp64")),
                    cg=rng.choice(("fp64", "mixed")), internal=0, steps=4)
    if kind == "ensemble":
        return dict(kind="ensemble", nb=rng.randint(3, 24), kc=rng.randint(2, 6),
                    store=rng.choice(("fp32", "fp64")), cg="fp64", steps=4)
    if kind == "adjoint":
        return dict(kind="adjoint", nx=rng.randint(40, 180), kc=rng.randint(2, 8),
                    nsrc=rng.randint(2, 8), nobs=rng.randint(10, 40), nsteps=12, every=4, ckpt=6,
                    store=rng.choice(("fp32", "fp64")))
    return dict(kind="restart", nx=rng.randint(24, 90), ny=rng.randint(20, 75),
                kc=rng.randint(2, 8))


# ------------------------------------------------------------------ inputs

def _field(rng, shape, lo, hi):
    """A smooth random field: a coarse grid of values, interpolated."""
    ny, nx = shape
    my, mx = max(4, ny // 24 + 2), max(4, nx // 24 + 2)
    z = rng.uniform(lo, hi, (my, mx))
    y, x = np.linspace(0, my - 1.001, ny), np.linspace(0, mx - 1.001, nx)
    j, i = y.astype(int), x.astype(int)
    fy, fx = (y - j)[:, None], (x - i)[None, :]
    a = z[j][:, i] * (1 - fx) + z[j][:, i + 1] * fx
    b = z[j + 1][:, i] * (1 - fx) + z[j + 1][:, i + 1] * fx
    return a * (1 - fy) + b * fy


def _flowing(c, seed, wind=1e-5, floor=0.0):
    """A surface in motion: a free-surface perturbation of some cm, external
    flows of some cm/s and a weak wind on the case's cells; cells and faces
    shallower than `floor` stay at rest."""
    rng = np.random.default_rng(seed + 7)
    g, h = c.grid, c.h
    L = np.arange(2, g.LA + 1) - 1
    jj, ii = g.JL[L] - 1, g.IL[L] - 1
    shape = (g.JC, g.IC)
    eta = 0.05 * (_field(rng, shape, -1, 1) + 0.2 * rng.standard_normal(shape))
    dx = float(c.meta["dx"])
    u, v = _field(rng, shape, -0.05, 0.05), _field(rng, shape, -0.05, 0.05)
    deep = h["HP"] > floor
    h["HP"][L] += eta[jj, ii] * deep[L]
    h["H1P"][:] = h["HP"]
    h["H2P"][:] = h["HP"]
    h["P"][L] = G * (h["HP"][L] + h["BELV"][L])
    h["P1"][:] = h["P"]
    grids.update_depth_arrays(g, h)
    grids.layer_depths(g, h, c.k)
    c.k["H1PK"][:] = c.k["HPK"]
    for a, f, hh, s, d in (("UHDYE", u, "HU", "SUB", "LWC"), ("VHDXE", v, "HV", "SVB", "LSC")):
        both = deep[L] & deep[g.maps[d][L] - 1]
        h[a][L] = f[jj, ii] * dx * h[hh][L] * h[s][L] * both
        h["UHDY1E" if a == "UHDYE" else "VHDX1E"][:] = h[a]
    h["UHE"][:] = h["UHDYE"] * h["DYIU"]
    h["VHE"][:] = h["VHDXE"] * h["DXIV"]
    h["TSX"][L] = wind * _field(rng, shape, -1, 1)[jj, ii]
    h["TSY"][L] = wind * _field(rng, shape, -1, 1)[jj, ii]
    for a, b in (("H1U", "HU"), ("H1V", "HV"), ("H1UI", "HUI"), ("H1VI", "HVI")):
        h[a][:] = h[b]
    return c


def _sheared(c, seed):
    """The internal-mode arrays with a sheared flow and viscosities of
    1e-4..1e-2 m2/s."""
    rng = np.random.default_rng(seed + 9)
    grids.add_internal_mode(c, av=1e-3)
    g, k = c.grid, c.k
    KC = g.KC
    L = np.arange(2, g.LA + 1) - 1
    f = 1.0 + 0.4 * np.cos(np.pi * (np.arange(KC) + 0.5) / KC)
    f = f / f.mean()
    for lvl in ("", "1"):
        for a in ("UHDYF", "VHDXF", "UHDY", "VHDX", "U", "V"):
            k[a + lvl][:KC] *= f[:, None]
    for a in ("AVUI", "AVVI"):
        for K in range(KC - 1):
            k[a][K, L] = 1.0 / np.exp(rng.uniform(math.log(1e-4), math.log(1e-2), len(L)))
    for a in ("VU", "V1U"):
        c.h[a][:] = k["V"][0] * 0.5
    for a in ("UV", "U1V"):
        c.h[a][:] = k["U"][0] * 0.5
    return c


def _lake(case, seed):
    # the shore belongs to the case; the bed and the state to the seed
    m = grids.lake_mask(case["nx"], case["ny"], 1001)
    rng = np.random.default_rng(seed)
    g = grids.build_grid(m, 1)
    h, k, w = grids._empty_arrays(g)
    grids.fill_geometry(g, h, k, w, 100.0, np.ones(1))
    L = np.arange(2, g.LA + 1) - 1
    jj, ii = g.JL[L] - 1, g.IL[L] - 1
    dep = _field(rng, m.shape, 4.0, 36.0)[jj, ii] + rng.uniform(-2, 4, len(L))
    h["BELV"][L] = -dep
    h["HP"][L] = dep
    c = grids.Case(name="lake", grid=g, h=h, k=k, w=w, consts=[], dt=10.0,
                   meta=dict(seed=seed, dx=100.0))
    return _flowing(c, seed)


def _constituents(c, nc, seed):
    """The first nc constituents of a case, with its source table."""
    c.consts = c.consts[:nc]
    s = c.sources
    s["cqs"], s["csert"] = s["cqs"][:, :, :nc].copy(), s["csert"][:, :, :nc].copy()
    return c


def _inputs(case, seed):
    """The case's arrays on the host (a grids.Case) and its context options."""
    kind = case["kind"]
    mixed = case.get("cg") == "mixed"
    opt = dict(cg_mode=lib.CG_MIXED if mixed else lib.CG_FP64, cg_rel_tol=1e-10, RSQM=0.0,
               ITERM=2000)
    if "store" in case:
        opt["store"] = lib.STORE_FP32 if case["store"] == "fp32" else lib.STORE_FP64
    if kind == "external" and case["isdry"]:
        c = grids.drying_basin(case["nx"], case["ny"], 1, seed=seed, dx=100.0)
        rng = np.random.default_rng(seed)
        g = c.grid
        L = np.arange(2, g.LA + 1) - 1
        rough = _field(rng, (g.JC, g.IC), -0.15, 0.15)[g.JL[L] - 1, g.IL[L] - 1]
        c.h["BELV"][L] += rough
        hp = np.maximum(c.h["HP"][L] - rough, 0.1)
        for a in ("HP", "H1P", "H2P"):
            c.h[a][L] = hp
        c.h["P"][L] = G * (hp + c.h["BELV"][L])
        c.h["P1"][:] = c.h["P"]
        grids.update_depth_arrays(g, c.h)
        grids.layer_depths(g, c.h, c.k)
        c.k["H1PK"][:] = c.k["HPK"]
        c.consts, c.conc_bc, c.sources, c.manning_n = [], None, None, None
        opt.update(ISDRY=case["isdry"])
        return _flowing(c, seed, floor=0.6), opt, None
    if kind == "external":
        return _lake(case, seed), opt, None
    if kind == "hydro":
        c = grids.tidal_basin(case["nx"], case["ny"], case["kc"], seed=seed, depth=(5.0, 20.0))
        c = _sheared(_flowing(c, seed), seed)
        c.manning_n = None
        # the boundary cell lists stay (CALUVW's open faces read them)
        return c, opt, None
    if kind == "transport":
        c = grids.transport_case(case["nx"], case["ny"], case["kc"], seed=seed,
                                 isadac=case["adac"], isfct=case["adac"])
        return _constituents(c, case["nconst"], seed), opt, None
    if kind in ("step", "restart"):
        c = grids.tidal_basin(case["nx"], case["ny"], case["kc"], seed=seed)
        c = _flowing(c, seed)
        if kind == "restart" or case["internal"]:
            c = _sheared(c, seed)
        return c, opt, None
    if kind == "ensemble":
        # the basins belong to the case; their state to the seed
        members = [_flowing(grids.ensemble_member(b, case["kc"]), seed + b)
                   for b in range(case["nb"])]
        c, first = grids.concat_basins(members)
        return c, opt, first
    raise ValueError(kind)


# ----------------------------------------------------------- device views

class _Array:
    """A device array of a context, as torch sees foreign memory; it keeps
    its owner alive."""

    def __init__(self, owner, ptr, shape, strides, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, strides=strides,
                                             typestr=typestr, version=2)


class _Views:
    """Torch views of a context's arrays by name, wet cells only.  The time
    levels swap buffers, so a view is made once per buffer and found by its
    address."""

    def __init__(self, ctx):
        self.ctx, self.seen = ctx, {}
        self.p, self.n = lib.C.c_void_p(), lib.C.c_int64()
        self.s = ctx.params.store

    def __call__(self, name):
        ctx, i = self.ctx, abi.ARRAY_IDS[name]
        ctx._check(ctx.lib.efdc_device_ptr(ctx.h, i, lib.C.byref(self.p), lib.C.byref(self.n)))
        key = (self.p.value, name)
        t = self.seen.get(key)
        if t is None:
            cls, g = abi.shape_class(name), ctx.grid
            wide = cls == "h" or i >= abi.ARRAY_IDS["STBX"] or self.s == lib.STORE_FP64
            z, ty = (8, "<f8") if wide else (4, "<f4")
            n = g.LA - 1
            if cls == "h":
                a = _Array(ctx, self.p.value + z, (n,), None, ty)
            else:
                a = _Array(ctx, self.p.value + z, (g.KC + (cls == "w"), n),
                           (z * self.n.value, z), ty)
            t = self.seen[key] = torch.as_tensor(a, device="cuda")
        return t


def _up(n):
    return (n + 255) & ~255


def _snapshot(ctx, case, cc):
    """A snapshot buffer and the views of the constituents in it."""
    g = ctx.grid
    pitch = lib.C.c_int64()
    p = lib.C.c_void_p()
    ctx._check(ctx.lib.efdc_device_ptr(ctx.h, abi.ARRAY_IDS["HPK"], lib.C.byref(p),
                                       lib.C.byref(pitch)))
    pitch = pitch.value
    z, dt = (4, torch.float32) if ctx.params.store == lib.STORE_FP32 else (8, torch.float64)
    buf = torch.zeros(ctx.state_bytes(), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    con = NH * _up(8 * g.LCM) + NK * _up(z * pitch * g.KC) + NW * _up(z * pitch * (g.KC + 1))
    plane = _up(z * pitch * g.KC)

    def layers(a):
        return buf[a:a + z * pitch * g.KC].view(dt).view(g.KC, pitch)[:, 1:g.LA]

    views = [layers(con + 2 * c * plane) for c in range(len(cc.consts))]
    old = [layers(con + (2 * c + 1) * plane) for c in range(len(cc.consts))]
    # the snapshot is where the model's checkpoints keep the constituents
    ctx.state_save(buf.data_ptr())
    ctx.synchronize()
    for v, x in zip(views, cc.consts):
        want = torch.from_numpy(x["con"][:1, 1:g.LA]).to(dt)
        if not torch.equal(v[:1].cpu(), want):
            raise RuntimeError("the snapshot does not hold the constituents where expected")
    hv = {}
    for name in EXT_OUT:
        a = abi.ARRAY_IDS[name] * _up(8 * g.LCM)
        hv[name] = buf[a:a + 8 * g.LCM].view(torch.float64)[1:g.LA]
    for name in STEP_OUT_K:
        hv[name] = layers(NH * _up(8 * g.LCM) +
                          (abi.ARRAY_IDS[name] - abi.ARRAY_IDS["HPK"]) * plane)
    return buf, dict(con=views, con1=old), hv


def prepare(case, seed):
    kind = case["kind"]
    if kind == "adjoint":
        c, obs, data, loads = _adjoint_inputs(case, seed)
        prob = adjoint.DyeMisfit(c, nsteps=case["nsteps"], obs_L=obs, obs_every=case["every"],
                                 data=data, ckpt=case["ckpt"],
                                 store=lib.STORE_FP32 if case["store"] == "fp32"
                                 else lib.STORE_FP64)
        return dict(kind=kind, prob=prob, loads=loads)
    c, opt, first = _inputs(case, seed)
    ctx = lib.Context(c.grid, **opt)
    ctx.upload_case(c)
    if first is not None:
        ctx.set_segments(first)
    s = dict(kind=kind, ctx=ctx, dt=c.dt, n=0, steps=case.get("steps", 1))
    if kind == "external":
        s["names"] = EXT_OUT + (("SUB", "SVB") if case["isdry"] else ())
        s["views"] = _Views(ctx)
    elif kind == "hydro":
        s["views"] = _Views(ctx)
        s["uvw"] = dict(wind=1)
        s["names"] = UVW_OUT_H + UVW_OUT_K + ("W", "W2")
    elif kind == "restart":
        s["opts"] = _restart_opts(case, c, seed)
        s["n"] = 720
    else:
        s["buf"], s["con"], s["h"] = _snapshot(ctx, case, c)
        s["internal"] = bool(case.get("internal"))
        s["levels"] = kind != "transport"
    ctx.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "adjoint":
        J, gl, gn, _ = s["prob"].gradient(s["loads"])
        return dict(J=J, loads=gl, manning=gn)
    ctx, dt = s["ctx"], s["dt"]
    if kind == "external":
        s["n"] += 1
        ctx.calpuv2c(dt, s["n"])
        return {a: s["views"](a) for a in s["names"]}
    if kind == "hydro":
        s["n"] += 1
        ctx.calpuv2c(dt, s["n"])
        ctx.caluvw(dt, s["n"], **s["uvw"])
        return {a: s["views"](a) for a in s["names"]}
    if kind == "restart":
        text = ctx.restart_text(s["n"], s["n"] * dt / 86400.0, **s["opts"])
        return np.frombuffer(text, np.uint8)
    for _ in range(s["steps"]):
        s["n"] += 1
        if kind == "transport":
            ctx.calconc(dt, s["n"])
        else:
            ctx.step(dt, s["n"], internal=s["internal"])
    ctx.state_save(s["buf"].data_ptr())
    return dict(s["con"], h=s["h"] if s["levels"] else None)


# -------------------------------------------------------------- the limits

def work(case):
    """Bytes: every array a pass needs and every array it leaves, once per
    step, in the width that the storage option gives it; operations: those
    of the formulas, with the iterations such solves take."""
    kind = case["kind"]
    s = 4 if case.get("store") == "fp32" else 8
    kc = case.get("kc", 1)
    ext = 8 * (33 + 28) + 16           # CALPUV2C per cell: arrays in and out, maps
    if kind == "external":
        n = case["nx"] * case["ny"] * (1.0 if case["isdry"] else 0.67)
        return dict(bytes=n * ext, flops=n * (150 + 20 * 24))
    if kind == "hydro":
        n = case["nx"] * case["ny"]
        uvw = 8 * (kc * 20 + kc * 13) + s * kc * 9 + 8 * 40
        return dict(bytes=n * (ext + uvw), flops=n * (150 + 20 * 24 + 120 * kc))

    def tran(nc):
        return kc * s * (6 + 2 * nc) + 40

    if kind == "transport":
        n = case["nx"] * case["ny"]
        nc = case["nconst"]
        more = nc * kc * s * 4 if case["adac"] else 0
        snap = s * kc * (NK + NW + 2 * nc) + 8 * NH
        return dict(bytes=n * (case["steps"] * (tran(nc) + more) + snap),
                    flops=n * case["steps"] * kc * nc * (100 if case["adac"] else 30))
    if kind in ("step", "ensemble"):
        n = case["nx"] * case["ny"] if kind == "step" else case["nb"] * 16000
        snap = s * kc * (NK + NW + 4) + 8 * NH
        uvw = 8 * (kc * 20 + kc * 13) + s * kc * 9 + 8 * 40
        per = ext + tran(2) + (uvw if case.get("internal") else 7 * s * kc + 80)
        return dict(bytes=n * (case["steps"] * per + snap),
                    flops=n * case["steps"] * (150 + 20 * 24 + 60 * kc))
    if kind == "adjoint":
        n = case["nx"] ** 2
        fwd = ext + tran(2) + 7 * s * kc + 80
        snap = s * kc * (NK + NW + 4) + 8 * NH
        rev = kc * (s * 8 + 8 * 4) + 8 * 60
        per = 2 * fwd + 2 * snap + rev
        return dict(bytes=n * case["nsteps"] * per, flops=n * case["nsteps"] * (1500 + 150 * kc))
    n = case["nx"] * case["ny"]        # restart: FP64 values in, 17 characters each out
    vals = 5 + 4 + 4 * kc + 5 * (kc + 1) + 4 * kc + 1 + kc
    return dict(bytes=n * vals * 25.0, flops=n * vals * 60.0)


def tolerance(case):
    kind = case["kind"]
    if kind == "restart":
        return "exact"
    f32 = case.get("store") == "fp32"
    # about four times what the path is off FP64 torch: FP32 storage rounds
    # each value once a step (1e-7 seen), FP64 sums differ in their order, and
    # the solves stop at a relative residual of 1e-10 (up to 1e-10 seen in
    # the flows, more after some steps, and where a solve ends one iteration
    # sooner or later)
    if kind == "transport":
        return dict(rel=5e-7, max=2e-5) if f32 else dict(rel=1e-13, max=1e-11)
    if kind == "external":
        return dict(rel=1e-9, max=1e-6)
    if kind == "adjoint":
        return dict(rel=3e-6, max=1e-3) if f32 else dict(rel=1e-8, max=1e-5)
    return dict(rel=1e-6, max=1e-4) if f32 else dict(rel=1e-8, max=1e-5)


# ------------------------------------------------- other inputs of a kind

def _restart_opts(case, c, seed):
    rng = np.random.default_rng(seed + 3)
    lcm, kc, hp = c.grid.LCM, c.grid.KC, c.h["HP"]
    mo = [x["mo"] for x in c.consts]
    return dict(isco=[0, 1, 0, 1, 0, 0, 0, 0, 0], istran=[0, 1, 0, 1, 0, 0, 0, 0, 0],
                slots=(mo.index(1), -1, mo.index(3)), keep_nlo=True,
                hwq=hp.copy(), h2wq=hp.copy(),
                qq=rng.uniform(1e-8, 1e-3, (kc + 1, lcm)),
                qq1=rng.uniform(1e-8, 1e-3, (kc + 1, lcm)),
                qql=rng.uniform(1e-9, 1e-4, (kc + 1, lcm)),
                qql1=rng.uniform(1e-9, 1e-4, (kc + 1, lcm)),
                dml=rng.uniform(0.0, 1.0, (kc + 1, lcm)))


def _adjoint_inputs(case, seed):
    c, obs = grids.adjoint_case(case["nx"], case["kc"], case["nsrc"], case["nobs"], seed=seed)
    c = _flowing(c, seed)
    rng = np.random.default_rng(seed + 5)
    nsteps, every = case["nsteps"], case["every"]
    loads = rng.uniform(0.0, 5.0, (nsteps, case["nsrc"]))
    # observed layer-mean dye of a window this short: about load * time / volume
    scale = 2.5 * nsteps * c.dt / (1e4 * 10.0 * 10)
    data = rng.uniform(0.0, scale, (nsteps // every, len(obs)))
    return c, obs, data, loads


# ------------------------------------------------------------ in 64 bits

class _Solve(torch.autograd.Function):
    """x of the 5-point system, by Jacobi-PCG from x0; its reverse solves
    the same (symmetric) system."""

    @staticmethod
    def forward(f, cc, cs, cw, ce, cn, b, x0, m, wet):
        x = _pcg(cc, cs, cw, ce, cn, b, x0, m, wet)
        f.save_for_backward(cc, cs, cw, ce, cn, x)
        f.m, f.wet = m, wet
        return x

    @staticmethod
    def backward(f, gx):
        cc, cs, cw, ce, cn, x = f.saved_tensors
        m = f.m
        gx = torch.where(f.wet, gx, torch.zeros_like(gx))
        mu = _pcg(cc, cs, cw, ce, cn, gx, torch.zeros_like(gx), m, f.wet)
        return (-mu * x, -mu * x[m["S"]], -mu * x[m["W"]], -mu * x[m["E"]], -mu * x[m["N"]], mu,
                None, None, None)


def _pcg(cc, cs, cw, ce, cn, b, x, m, wet):
    ci = torch.where(wet, 1.0 / torch.where(wet, cc, torch.ones_like(cc)), torch.zeros_like(cc))

    def mul(p):
        return torch.where(wet, cc * p + cs * p[m["S"]] + cw * p[m["W"]] + ce * p[m["E"]] +
                           cn * p[m["N"]], torch.zeros_like(p))

    def dot(p, q):
        return torch.dot(p, q)

    x = torch.where(wet, x, torch.zeros_like(x))
    b = torch.where(wet, b, torch.zeros_like(b))
    stop = 1e-30 * float(dot(b * ci, b))
    for _ in range(3):                    # restarted: the true residual each time
        r = b - mul(x)
        z = ci * r
        p, rz = z, dot(r, z)
        for it in range(400):
            if it % 8 == 0 and float(rz) <= stop:
                break
            ap = mul(p)
            a = rz / dot(p, ap)
            x, r = x + a * p, r - a * ap
            z = ci * r
            new = dot(r, z)
            p, rz = z + (new / rz) * p, new
    return x


class _Model:
    """The steps in FP64 torch, on the case's arrays."""

    def __init__(self, c, isdry=0, hdry=0.2):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.c, g = c, c.grid
        self.dt, self.KC, self.LA = c.dt, g.KC, g.LA
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
        self.t = t
        self.h = {k: t(v).clone() for k, v in c.h.items()}
        self.k = {k: t(v[:g.KC]).clone() for k, v in c.k.items()}
        self.w = {k: t(v[:g.KC + 1]).clone() for k, v in c.w.items()}
        self.m = {d: t(c.grid.maps[n].astype(np.int64) - 1)
                  for d, n in dict(W="LWC", E="LEC", S="LSC", N="LNC", NW="LNWC",
                                   SE="LSEC").items()}
        self.con = [t(x["con"][:g.KC]).clone() for x in c.consts]
        wet = torch.zeros(g.LCM, dtype=torch.bool, device=dev)
        wet[1:g.LA] = True
        self.wet = wet
        self.zero = torch.zeros(g.LCM, dtype=torch.float64, device=dev)
        self.nman = None if c.manning_n is None else t(c.manning_n)
        self.isdry, self.hdry = isdry, hdry
        side = c.open_bc["side"][0] if c.open_bc is not None else None
        self.bw = t(side["L"].astype(np.int64) - 1) if side is not None else None
        self.pcb = t(np.asarray(side["pcb"]).reshape(-1)) if side is not None else None
        self.clo = self.nlo = None

    def only(self, a):
        return torch.where(self.wet, a, torch.zeros_like(a))

    def set(self, **kw):
        for k, v in kw.items():
            self.h[k] = self.only(v)

    # --- closure, CALPUV2C
    def pre(self):
        if self.nman is None:
            return
        h, one = self.h, torch.ones_like(self.zero)
        for tb, q, hh in (("TBX", "UHE", "HU"), ("TBY", "VHE", "HV")):
            d = torch.where(self.wet, h[hh], one)
            u = h[q] / d
            h[tb] = self.only(G * self.nman ** 2 * u * torch.abs(u) / d ** (1.0 / 3.0))

    def puv(self, n):
        h, m, dt, wet = self.h, self.m, self.dt, self.wet
        d2 = 0.5 * dt
        p, e, nn, w, s = h["P"], m["E"], m["N"], m["W"], m["S"]
        fu = (h["UHDYE"] - d2 * h["SUB"] * h["HRUO"] * h["HU"] * (p - p[w]) +
              h["SUB"] * dt * h["DXIU"] * (h["DXYU"] * (h["TSX"] - h["TBX"]) + h["FCAXE"]))
        fv = (h["VHDXE"] - d2 * h["SVB"] * h["HRVO"] * h["HV"] * (p - p[s]) +
              h["SVB"] * dt * h["DYIV"] * (h["DXYV"] * (h["TSY"] - h["TBY"]) - h["FCAYE"]))
        fu, fv = self.only(fu), self.only(fv)
        sub1, svb1 = h["SUB"], h["SVB"]
        if self.isdry:
            self.set(SUB=h["SUBO"], SVB=h["SVBO"])
        u1, v1, h1 = h["UHDYE"], h["VHDXE"], h["HP"]
        self.set(UHDY1E=u1, VHDX1E=v1, P1=p, H1U=h["HU"], H1V=h["HV"], H1UI=h["HUI"],
                 H1VI=h["HVI"], H2P=h["H1P"], H1P=h1)
        self.k["H1PK"] = self.k["HPK"]
        fp1 = h["DXYP"] / dt * p - 0.5 * G * (u1[e] - u1 + v1[nn] - v1)
        iscdry = torch.zeros_like(wet)
        obdry = torch.zeros_like(wet)
        keep_cc = None
        for _ in range(500):
            sub, svb = h["SUB"], h["SVB"]
            a = sub * fu
            b = svb * fv
            fp = fp1 - 0.5 * G * (a[e] - a + b[nn] - b - 2.0 * h["QSUME"])
            cw = -0.5 * d2 * G * sub * h["HRUO"] * h["RCX"] * h["HU"]
            cs = -0.5 * d2 * G * svb * h["HRVO"] * h["RCY"] * h["HV"]
            ce, cn = cw[e], cs[nn]
            cc = h["DXYP"] / dt - cs - cw - ce - cn
            if self.bw is not None:       # clamped west cells
                bw = self.bw
                be = e[bw]
                z = torch.zeros_like(h["P"][bw])
                ph = PI2 * math.fmod(dt * n, float(self.c.open_bc["tcp"][0])) / \
                    float(self.c.open_bc["tcp"][0])
                val = self.pcb * math.cos(ph)
                low = 0.2 * self.hdry
                dry = ((val / G - low) < h["BELV"][bw]) | ((val / G - low) < h["BELV"][be])
                already = obdry[bw]
                val = torch.where(dry, (h["BELV"][bw] + low) * G, val)
                cet = torch.where(dry, z, 0.5 * d2 * G * h["HRUO"][be] * h["RCX"][be] *
                                  h["HU"][be])
                add = torch.where(already, z, cet * val)
                fp = fp.index_add(0, be, add)
                own = torch.where(already, fp[bw], h["DXYP"][bw] / dt * val)
                fp = fp.index_copy(0, bw, own)
                obdry = obdry.index_copy(0, bw, already | dry)
                cc = cc.index_copy(0, bw, h["DXYP"][bw] / dt)
                cw, cs = cw.index_copy(0, bw, z), cs.index_copy(0, bw, z)
                ce, cn = ce.index_copy(0, bw, z), cn.index_copy(0, bw, z)
                cw = cw.index_copy(0, be, z)
            x = _Solve.apply(cc, cs, cw, ce, cn, fp, p.detach(), m, wet)
            u = self.only(sub * (fu - d2 * h["HRUO"] * h["RCX"] * h["HU"] * (x - x[w])))
            v = self.only(svb * (fv - d2 * h["HRVO"] * h["RCY"] * h["HV"] * (x - x[s])))
            self.set(UHDYE=u, VHDXE=v, UHE=u * h["DYIU"], VHE=v * h["DXIV"])
            hp = h1 + d2 * h["DXYIP"] * (2.0 * h["QSUME"] - (u[e] + u1[e] - u - u1 + v[nn] +
                                                            v1[nn] - v - v1))
            if self.bw is not None:
                hp = hp.index_copy(0, self.bw, x[self.bw] / G - h["BELV"][self.bw])
            self.set(HP=hp)
            if not self.isdry:
                break
            fp1 = self._open_dry(iscdry, obdry, fp1, h1)
            p = self.only(G * (h["HP"] + h["BELV"]))
            if not (self._dry(iscdry) if self.isdry < 98 else self._rewet(iscdry, h1)):
                break
        hp = h["HP"]
        one = torch.ones_like(hp)
        self.set(P=G * (hp + h["BELV"]))
        a = h["DXYP"] * hp
        hu = (a + a[w]) * (0.5 / torch.where(wet, h["DXYU"], one))
        hv = (a + a[s]) * (0.5 / torch.where(wet, h["DXYV"], one))
        self.set(HU=hu, HV=hv, HPI=1.0 / torch.where(wet, hp, one),
                 HUI=1.0 / torch.where(wet, hu, one), HVI=1.0 / torch.where(wet, hv, one))

    def _close(self, cells, obc=None):
        """Close the four faces of the marked cells."""
        h, m = self.h, self.m
        for a, d in (("SUB", "E"), ("SVB", "N")):
            x = h[a].clone()
            x[cells] = 0.0
            x[m[d][cells]] = 0.0
            h[a] = self.only(x)
            if obc:
                q = h[obc[a]].clone()
                q[cells] = 0.0
                q[m[d][cells]] = 0.0
                h[obc[a]] = self.only(q)

    def _open_dry(self, iscdry, obdry, fp1, h1):
        h = self.h
        bw = self.bw
        hp, q = h["HP"][bw], h1[bw]
        go = (obdry[bw] | ((q < 0.9 * self.hdry) & (hp < q)) | (hp < 0.0)) & ~iscdry[bw]
        if not bool(go.any()):
            return fp1
        c = bw[go]
        new = torch.clamp(q[go], 0.1 * self.hdry, 0.9 * self.hdry)
        new = torch.where((hp[go] <= 0.0) & obdry[c], torch.full_like(new, 0.2 * self.hdry), new)
        h["HP"] = h["HP"].index_copy(0, c, new)
        iscdry[c] = True
        obdry[c] = True
        self._close(c, dict(SUB="UHDYE", SVB="VHDXE"))
        return fp1.index_copy(0, c, h["DXYP"][c] / self.dt * (new + h["BELV"][c]) * G)

    def _dry(self, iscdry):
        c = torch.nonzero(self.wet & (self.h["HP"] <= self.hdry)).flatten()
        again = bool((~iscdry[c]).any())
        iscdry[c] = True
        self._close(c)
        return again

    def _rewet(self, iscdry, h1):
        """ISDRY = 99, the cells in the order of L (each reads the faces that
        the cells before it have set)."""
        h, m = self.h, self.m
        n = lambda a: a.cpu().numpy()  # noqa: E731
        hp, h1, sub, svb = n(h["HP"]), n(h1), n(h["SUB"]).copy(), n(h["SVB"]).copy()
        so, vo, u, v = n(h["SUBO"]), n(h["SVBO"]), n(h["UHDYE"]), n(h["VHDXE"])
        mw, me, ms, mn = (n(m[d]) for d in "WESN")
        isc = n(iscdry).copy()
        hd, again = self.hdry, False
        for i in np.nonzero(n(self.wet) & (hp <= hd))[0]:
            e, nn = me[i], mn[i]
            was = (sub[i], sub[e], svb[i], svb[nn])
            dh = hp[i] - h1[i]
            if dh > 0.0:
                sub[i] = sub[e] = svb[i] = svb[nn] = 0.0
                if dh > (hd - h1[i]) * 0.01:
                    if so[i] > 0.5 and u[i] > 0 and hp[mw[i]] > 2 * hd:
                        sub[i] = so[i]
                    if so[e] > 0.5 and u[e] < 0 and hp[e] > 2 * hd:
                        sub[e] = so[e]
                    if vo[i] > 0.5 and v[i] > 0 and hp[ms[i]] > 2 * hd:
                        svb[i] = vo[i]
                    if vo[nn] > 0.5 and v[nn] < 0 and hp[nn] > 2 * hd:
                        svb[nn] = vo[nn]
                    now = (sub[i], sub[e], svb[i], svb[nn])
                    isc[i] = sum(now) < 0.5
                    again |= any(abs(a - b) > 0.5 for a, b in zip(now, was))
                elif not isc[i]:
                    isc[i], again = True, True
            elif hp[i] < 0.9 * hd or h1[i] < hd:
                sub[i] = sub[e] = svb[i] = svb[nn] = 0.0
                if not isc[i]:
                    isc[i], again = True, True
        self.set(SUB=self.t(sub), SVB=self.t(svb))
        iscdry.copy_(self.t(isc))
        return again

    def post(self):
        h, k = self.h, self.k
        z = k["DZC"]
        ub, vb = 0.5 * (h["UHDYE"] + h["UHDY1E"]), 0.5 * (h["VHDXE"] + h["VHDX1E"])
        k["UHDY2"], k["VHDX2"] = ub * z, vb * z
        k["HPK"] = h["HP"] * z
        k["HPKI"] = 1.0 / torch.where(self.wet, k["HPK"], torch.ones_like(z))

    # --- CALUVW
    def _faces(self, v):
        """Layer constants of the open faces (index K) and CERRU of open and
        closed ones."""
        KC = self.KC
        z = self.c.k["DZC"][:KC, 1]
        f = dict(sg=z, dzg=0.5 * (z[:-1] + z[1:]), cdzf=z[:-1] * z[1:] / (z[:-1] + z[1:]),
                 cdzu=-z[:-1] / (z[:-1] + z[1:]), cdzl=-z[1:] / (z[:-1] + z[1:]),
                 cdzm=0.5 * z[:-1] * z[1:], cdzd=np.cumsum(z)[:-1])
        f["cdzr"] = (np.cumsum(z)[:-1] - 1.0) * f["dzg"] * f["cdzl"][0]
        f["cerr"] = (1.0 / (1.0 - z)) / np.sum(1.0 / (1.0 - z)) * KC
        return f

    def uvw(self, wind):
        h, k, w, m, dt, KC = self.h, self.k, self.w, self.m, self.dt, self.KC
        KS = KC - 1
        e, nn = m["E"], m["N"]
        for a in ("UHDYF", "VHDXF", "UHDY", "VHDX", "U", "V"):
            k[a + "1"] = k[a]
        w["W1"] = w["W"]
        if KC == 1:
            raise NotImplementedError
        ek = [self.only(k["DZC"][:KS] * (h[a] - h[a][d])) for a, d in (("UHDYE", e),
                                                                        ("VHDXE", nn))]
        one = torch.ones_like(h["HP"])
        for q, (F, Q, V, V1, VX, V1X, E, EH, H, H1, HI, S, SO, ST, TS, AV, DY, DI) in enumerate((
                ("UHDYF", "UHDY", "U", "U1", "VU", "V1U", "UHDYE", "UHE", "HU", "H1U", "HUI",
                 "SUB", "SUBO", "STBX", "TSX", "AVUI", "DYU", "DYIU"),
                ("VHDXF", "VHDX", "V", "V1", "UV", "U1V", "VHDXE", "VHE", "HV", "H1V", "HVI",
                 "SVB", "SVBO", "STBY", "TSY", "AVVI", "DXV", "DXIV"))):
            f = self._faces(q)
            op = h[SO] > 0.0
            s3 = k["SUB3D" if q == 0 else "SVB3D"]
            on = op.to(torch.float64)
            q1 = torch.sqrt(k[V1][0] ** 2 + h[V1X] ** 2)
            q2 = torch.sqrt(k[V][0] ** 2 + h[VX] ** 2)
            rc = h[ST] * torch.sqrt(q1 * q2)
            d = [on * f["cdzf"][K] * h[H1] * (k[V1][K + 1] - k[V1][K]) / dt for K in range(KS)]
            if wind:
                d[KS - 1] = d[KS - 1] - on * f["cdzu"][KS - 1] * h[TS]
            cu, uu = [None] * KS, [None] * KS
            av = k[AV]
            for K in range(KS):
                cl, cup = on * f["cdzl"][K], on * f["cdzu"][K]
                cm = 1.0 + on * f["cdzm"][K] / dt * h[H] * av[K]
                d[K] = s3[K] * d[K]
                if K:
                    eu = 1.0 / (cm - cl * cu[K - 1])
                    d[K] = (d[K] - cl * d[K - 1]) * eu
                    uu[K] = -cl * uu[K - 1] * eu
                else:
                    eu = 1.0 / cm
                    d[K] = (d[K] - cl * rc * h[EH] * h[HI]) * eu
                    uu[K] = eu
                cu[K] = cup * eu
            for K in range(KS - 2, -1, -1):
                d[K] = d[K] - cu[K] * d[K + 1]
                uu[K] = uu[K] - cu[K] * uu[K + 1]
            aa, bb = torch.zeros_like(one), one
            for K in range(KS):
                cr = on * f["cdzr"][K] * rc * av[K]
                aa, bb = aa + cr * d[K], bb + cr * uu[K]
            aa = aa / bb
            dzg = [on * f["dzg"][K] for K in range(KS)]
            d = [s3[K] * dzg[K] * h[H] * av[K] * (d[K] - aa * uu[K]) for K in range(KS)]
            eh = h[EH]
            for K in range(KS):
                eh = eh + on * f["cdzd"][K] * d[K]
            fl = [None] * KC
            fl[KS] = eh * h[S]
            for K in range(KS - 1, -1, -1):
                fl[K] = s3[K] * (fl[K + 1] - d[K])
            fl = [x * h[DY] for x in fl]
            tv = sum(fl[K] * on * f["sg"][K] for K in range(KC)) - h[E]
            cerr = [torch.where(op, f["cerr"][K] * one, one) for K in range(KC)]
            fl = torch.stack([self.only(fl[K] - tv * cerr[K]) for K in range(KC)])
            sg = torch.stack([on * f["sg"][K] for K in range(KC)])
            k[F], k[Q] = fl, self.only(fl * sg)
            k[V] = self.only(fl * h[HI] * h[DI])
            h[EH] = self.only((fl * sg).sum(0) * h[DI])
        k1 = [k["UHDYEK"][:KS], k["VHDXEK"][:KS]]   # levels of the step before
        W = [torch.zeros_like(one)]
        for K in range(KS):
            a = 0.0
            for q, (Q, dd) in enumerate((("UHDY", e), ("VHDX", nn))):
                for x in (k[Q][K], k[Q + "1"][K]):
                    a = a + x[dd] - x
                a = a + ek[q][K] + k1[q][K]
            W.append(self.only(W[-1] - 0.5 * h["DXYIP"] * a +
                               (k["QSUM"][K] - k["DZC"][K] * h["QSUME"]) * h["DXYIP"]))
        W = torch.stack(W + [torch.zeros_like(one)])
        k["UHDYEK"], k["VHDXEK"] = (torch.cat([x, o[KS:]]) for x, o in
                                    zip(ek, (k["UHDYEK"], k["VHDXEK"])))
        bw, be = self.bw, e[self.bw]
        W[:, bw] = 0.0
        b2 = e[be]
        fl = k["UHDYF"].clone()
        fl[:, be] = fl[:, b2] - h["UHDYE"][b2] + h["UHDYE"][be]
        sg = self.t(self._faces(0)["sg"])[:, None]
        qq, u = k["UHDY"].clone(), k["U"].clone()
        qq[:, be] = fl[:, be] * sg
        u[:, be] = fl[:, be] / (h["HU"][be] * h["DYU"][be])
        W[:, be] = 0.0
        k["UHDYF"], k["UHDY"], k["U"] = fl, qq, u
        # interface K of the layer arrays' count, as the model keeps it
        w["W"] = torch.cat([W[:KS + 1], w["W"][KS + 1:]])
        for a in ("UHDYF", "VHDXF"):
            k[a + "2"] = 0.5 * (k[a] + k[a + "1"])
        for a, b in (("UHDY", "UHDY2"), ("VHDX", "VHDX2"), ("U", "U2"), ("V", "V2")):
            k[b] = 0.5 * (k[a] + k[a + "1"])
        w["W2"] = torch.cat([w["W2"][:1], 0.5 * (w["W"][1:] + w["W1"][1:])])
        te, tn = k["UHDY2"].sum(0), k["VHDX2"].sum(0)
        hp = h["H1P"] + dt * h["DXYIP"] * (h["QSUME"] + te - te[e] + tn - tn[nn])
        hp = hp.index_copy(0, bw, h["P"][bw] / G - h["BELV"][bw])
        self.set(HP=hp, HPI=1.0 / torch.where(self.wet, hp, one))
        k["HPK"] = h["HP"] * k["DZC"]
        k["HPKI"] = 1.0 / torch.where(self.wet, k["HPK"], torch.ones_like(k["HPK"]))
        hp = h["HP"]
        u, v = k["U"][0], k["V"][0]
        uv = self.only((hp * u)[m["SE"]] + (hp * u)[m["S"]] + (hp * u)[e] + hp * u) / \
            (1.0 + h["SUB"][e] + h["SUB"][m["S"]] + h["SUB"][m["SE"]]) * h["HVI"]
        vu = self.only((hp * v)[m["NW"]] + (hp * v)[m["W"]] + (hp * v)[nn] + hp * v) / \
            (1.0 + h["SVB"][nn] + h["SVB"][m["W"]] + h["SVB"][m["NW"]]) * h["HUI"]
        self.set(U1V=h["UV"], V1U=h["VU"])
        self.set(UV=uv, VU=vu)

    # --- CALCONC
    def tran(self, niter, cqs=None):
        h, k, m, dt, KC = self.h, self.k, self.m, self.dt, self.KC
        e, nn, w_, s_ = m["E"], m["N"], m["W"], m["S"]
        src = self.c.sources
        cqs = self.t(np.asarray(src["cqs"])) if cqs is None else cqs
        lq = self.t(src["LQS"].astype(np.int64) - 1)
        qss = self.t(np.asarray(src["qss"]))
        u, v = self.only(k["UHDY2"]), self.only(k["VHDX2"])
        wv = self.w["W2"][1:KC]
        z1 = torch.zeros_like(self.zero)[None]
        fac = self._factors()
        for c, x in enumerate(self.c.consts):
            old = self.con[c]
            fu = u * torch.where(u >= 0, old[:, w_], old)
            fv = v * torch.where(v >= 0, old[:, s_], old)
            fw = torch.cat([z1, wv * torch.where(wv >= 0, old[:-1], old[1:]), z1])
            q = torch.clamp(qss, min=0.0) * cqs[:, :, c] + \
                torch.clamp(qss, max=0.0) * old[:, lq].T
            fq = torch.zeros_like(old).index_add(1, lq, q.T.contiguous())
            new = (old * k["H1PK"] + dt * ((fq + fu - fu[:, e] + fv - fv[:, nn]) * h["DXYIP"] +
                                           (fw[:-1] - fw[1:]))) * k["HPKI"]
            new = self.only(new)
            if self.c.conc_bc is not None:
                new = self._open_conc(c, x, old, new, u, fu, niter)
            if x["isadac"]:
                new = self._adac(old, new, u, v, wv)
            # vertical diffusion
            if KC > 1:
                eeb, ccl, vcu = fac
                y = [new[0] * eeb[0]]
                for K in range(1, KC):
                    y.append((new[K] - ccl[K] * y[-1]) * eeb[K])
                out = [y[-1]]
                for K in range(KC - 2, -1, -1):
                    out.append(y[K] - vcu[K] * out[-1])
                new = torch.stack(out[::-1])
            if x["wset"] > 0:
                ws, sed, fl = x["wset"], [None] * KC, 0.0
                for K in range(KC - 1, 0, -1):
                    wl = dt * k["HPKI"][K]
                    sed[K] = (torch.clamp(new[K], min=0.0) - fl * wl) / (1.0 + ws * wl)
                    fl = -ws * sed[K]
                wl = dt * k["HPKI"][0]
                sed[0] = (torch.clamp(new[0], min=0.0) + (x["wese"] - fl) * wl) / \
                    (1.0 + x["probdep"] * ws * wl)
                new = torch.stack(sed)
            self.con[c] = self.only(new)

    def _factors(self):
        k, hpi, dt, KC = self.k, self.h["HPI"], self.dt, self.KC
        if KC == 1:
            return None
        ab, up, lo = k["AB"], k["CDZKK"], k["CDZKMK"]
        eeb, ccl, vcu = [], [], []
        for K in range(KC):
            a = -dt * lo[K] * hpi * ab[K - 1] if K else 0.0
            b = -dt * up[K] * hpi * ab[K] if K < KC - 1 else 0.0
            ccl.append(a)
            eeb.append(1.0 / (1.0 - a - b - (a * vcu[K - 1] if K else 0.0)))
            vcu.append(b * eeb[K])
        return eeb, ccl, vcu

    def _open_conc(self, c, x, old, new, u, fu, niter):
        """The west concentration boundary with its recovery ramp."""
        b = self.c.conc_bc["side"][1]
        bw = self.t(b["L"].astype(np.int64) - 1)
        be = self.m["E"][bw]
        KC, nc = self.KC, len(self.c.consts)
        if self.clo is None:
            z = torch.zeros(nc, KC, len(bw), dtype=torch.float64, device=bw.device)
            self.clo, self.nlo = list(z), list(z.clone())
        cb = self.t(np.asarray(b["cb"]))[:, :, c]
        cst = self.t(np.asarray(b["csert"]))[:, :, c].T
        wt = self.t(np.asarray(self.c.conc_bc["wtci"]))
        ts = self.t(np.asarray(b["ntscr"]).astype(np.float64))
        flow = u[:, be]
        out = flow <= 0.0
        c1 = old[:, bw]
        gone = torch.clamp(c1 + self.dt * (flow * c1 - fu[:, be]) * self.h["DXYIP"][bw] *
                           self.k["HPKI"][:, bw], min=0.0)
        if x["mo"] == 1:
            gone = torch.minimum(gone, (cb[:, 0] + cst[0])[None])
        cbt = wt[:, :1] * cb[:, 0] + wt[:, 1:] * cb[:, 1] + cst
        age = niter - self.nlo[c]
        ramp = torch.clamp(self.clo[c] + (cbt - self.clo[c]) * age / ts, min=0.0)
        val = torch.where(out, gone, torch.where(age >= ts, cbt, ramp))
        self.clo[c] = torch.where(out, val, self.clo[c])
        self.nlo[c] = torch.where(out, torch.full_like(self.nlo[c], float(niter)), self.nlo[c])
        return new.index_copy(1, bw, val)

    def _adac(self, old, con, u, v, wv):
        """Anti-diffusion with the flux limiter, on a closed basin."""
        h, k, m, dt, KC = self.h, self.k, self.m, self.dt, self.KC
        e, nn, w_, s_ = m["E"], m["N"], m["W"], m["S"]
        eps = 1.0e-6
        mx, mn = torch.maximum, torch.minimum
        z1 = torch.zeros_like(self.zero)[None]
        pos = self.only(torch.clamp(con, min=0.0))
        uu = self.only(k["U2"] * (pos - pos[:, w_]) * h["DXIU"])
        vv = self.only(k["V2"] * (pos - pos[:, s_]) * h["DYIV"])
        ww = torch.cat([z1, self.only(wv * (pos[1:] - pos[:-1]) * h["HPI"] *
                                      self.w["DZIG"][1:KC]), z1])
        wt = ww[1:] + ww[:-1]
        t = torch.abs(u) * (pos - pos[:, w_])
        t = t - 0.5 * dt * u * torch.where(
            u >= 0, vv[:, m["NW"]] + vv[:, w_] + wt[:, w_] + uu + uu[:, w_],
            vv[:, nn] + vv + wt + uu + uu[:, e])
        a = t / (pos + pos[:, w_] + eps)
        fu = self.only(torch.clamp(a, min=0) * pos[:, w_] + torch.clamp(a, max=0) * pos)
        t = torch.abs(v) * (pos - pos[:, s_])
        t = t - 0.5 * dt * v * torch.where(
            v >= 0, uu[:, s_] + uu[:, m["SE"]] + wt[:, s_] + vv[:, s_] + vv,
            uu + uu[:, e] + wt + vv[:, nn] + vv)
        a = t / (pos + pos[:, s_] + eps)
        fv = self.only(torch.clamp(a, min=0) * pos[:, s_] + torch.clamp(a, max=0) * pos)
        hor = uu + uu[:, e] + vv + vv[:, nn]
        t = torch.abs(wv) * (pos[1:] - pos[:-1])
        t = t - 0.5 * dt * wv * torch.where(wv >= 0, hor[:-1] + ww[1:-1] + ww[:-2],
                                            hor[1:] + ww[1:-1] + ww[2:])
        a = t / (pos[1:] + pos[:-1] + eps)
        fw = torch.cat([z1, self.only(torch.clamp(a, min=0) * pos[:-1] +
                                      torch.clamp(a, max=0) * pos[1:]), z1])
        src = torch.abs(k["QSUM"]) > 1e-8
        for K, L in torch.nonzero(src & self.wet).tolist():
            fu[K, L] = fv[K, L] = 0.0
            fu[K, e[L]] = 0.0
            fv[K, nn[L]] = 0.0
            fw[K + 1, L] = 0.0 if K < KC - 1 else fw[K + 1, L]
        hi = mx(pos, torch.clamp(old, min=0.0))
        lo = mn(pos, torch.clamp(old, min=0.0))
        hi, lo = self.only(hi), self.only(lo)
        cmax, cmin = hi, lo
        cmax = mx(cmax, torch.cat([hi[1:], hi[-1:]]))
        cmax = mx(cmax, torch.cat([hi[:1], hi[:-1]]))
        cmin = mn(cmin, torch.cat([lo[1:], lo[-1:]]))
        cmin = mn(cmin, torch.cat([lo[:1], lo[:-1]]))
        sx, sy = k["SUB3D"], k["SVB3D"]
        for d, sw in ((w_, sx), (e, sx[:, e]), (s_, sy), (nn, sy[:, nn])):
            cmax = mx(cmax, sw * hi[:, d])
            cmin = mn(cmin, sw * lo[:, d] + 1e6 * (1.0 - sw))
        up, um = torch.clamp(fu, min=0), torch.clamp(fu, max=0)
        vp, vm = torch.clamp(fv, min=0), torch.clamp(fv, max=0)
        wp, wm = torch.clamp(fw, min=0), torch.clamp(fw, max=0)
        di = dt * ((up - um[:, e] + vp - vm[:, nn]) * h["DXYIP"] + wp[:-1] - wm[1:]) * k["HPKI"]
        do = dt * ((up[:, e] - um + vp[:, nn] - vm) * h["DXYIP"] + wp[1:] - wm[:-1]) * k["HPKI"]
        di = torch.clamp(torch.where(di > 0, (cmax - pos) / (di + eps), di), max=1.0)
        do = torch.clamp(torch.where(do > 0, (pos - cmin) / (do + eps), do), max=1.0)
        di, do = self.only(di), self.only(do)
        fu = mn(do[:, w_], di) * up + mn(di[:, w_], do) * um
        fv = mn(do[:, s_], di) * vp + mn(di[:, s_], do) * vm
        fw = torch.cat([z1, mn(do[:-1], di[1:]) * wp[1:-1] + mn(di[:-1], do[1:]) * wm[1:-1], z1])
        fu, fv, fw = self.only(fu), self.only(fv), self.only(fw)
        return self.only((con * k["HPK"] + dt * ((fu - fu[:, e] + fv - fv[:, nn]) * h["DXYIP"] +
                                                 fw[:-1] - fw[1:])) * k["HPKI"])

    def step(self, n, internal=False, cqs=None, wind=0):
        self.pre()
        self.puv(n)
        if internal:
            self.uvw(wind)
        else:
            self.post()
        self.tran(n, cqs)


def exact(case, seed):
    kind = case["kind"]
    if kind == "restart":
        return None
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    c, opt, _ = _inputs(case, seed)
    wet = slice(1, c.grid.LA)
    with torch.no_grad():
        m = _Model(c, isdry=case.get("isdry", 0))
        if kind == "external":
            m.puv(1)
            return {a: m.h[a][wet] for a in EXT_OUT + (("SUB", "SVB") if case["isdry"] else ())}
        if kind == "hydro":
            m.puv(1)
            m.uvw(1)
            out = {a: m.h[a][wet] for a in UVW_OUT_H}
            out.update({a: m.k[a][:, wet] for a in UVW_OUT_K})
            out.update({a: m.w[a][:, wet] for a in ("W", "W2")})
            return out
        for n in range(1, case["steps"] + 1):
            if kind == "transport":
                m.tran(n)
            else:
                m.step(n, internal=bool(case.get("internal")))
        h = None
        if kind != "transport":
            h = {a: m.h[a][wet] for a in EXT_OUT}
            h.update({a: m.k[a][:, wet] for a in STEP_OUT_K})
        return dict(con=[x[:, wet] for x in m.con], con1=[None] * len(m.con), h=h)


def _exact_adjoint(case, seed):
    c, obs, data, loads = _adjoint_inputs(case, seed)
    m = _Model(c)
    lo = m.t(loads).requires_grad_()
    nm = m.t(c.manning_n).clone().requires_grad_()
    m.nman = nm
    q = m.t(np.asarray(c.sources["qss"]).sum(axis=1))
    base = m.t(np.asarray(c.sources["cqs"], np.float64))
    y = m.t(data)
    ob = m.t(obs.astype(np.int64) - 1)
    dz = m.k["DZC"][:, ob]
    J = 0.0
    for n in range(1, case["nsteps"] + 1):
        dye = (lo[n - 1] / q)[:, None, None].expand(-1, base.shape[1], -1)
        m.step(n, cqs=torch.cat([base[:, :, :1], dye], dim=2))
        if n % case["every"] == 0:
            J = J + ((dz * m.con[1][:, ob]).sum(0) - y[n // case["every"] - 1]).square().sum()
    gl, gn = torch.autograd.grad(J, (lo, nm))
    return dict(J=float(J.detach()), loads=gl, manning=gn)
