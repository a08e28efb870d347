"""k_tran_lay (the default CALCONC column pass with mutual neighbour maps:
layers side by side in a workgroup, the vertical solve from LDS) against the
column kernels, whose bits it must give: layer counts at the edges of its
wave split (KC = 1, 2, 7, 8, 15) and of its LDS rule (21 and more: fewer
constituents a workgroup; 41: one workgroup a CU; 64: the most layers),
constituent counts that fill and that split the groups, open boundary,
source, settling, varying layer thickness, a dry mask, and the pass without
the vertical solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ctx(case, shape, **kw):
    from efdc_amd.lib import Context
    kw.setdefault("RSQM", 1e-22)
    kw.setdefault("ITERM", 2000)
    return Context(case.grid, tran_shape=shape, **kw).upload_case(case)


def _constituents(case, nc):
    """nc constituents: the case's, repeated; every third settles."""
    c = case.copy()
    base = c.consts
    c.consts = []
    for j in range(nc):
        x = dict(base[j % len(base)])
        x["con"] = x["con"] * (1.0 + 0.1 * j) + 0.01 * j
        x["con"][:, [0, -2, -1]] = 0.0
        x["con1"] = x["con"].copy()
        if j % 3 == 2:
            x.update(wset=2e-4 * (j + 1), probdep=0.7, wese=1e-6)
        else:
            x.update(wset=0.0)
        if x["is_dye"]:
            x["rkdye"] = (0.0, 1e-5, 1000.0)[j % 3]
        c.consts.append(x)
    pick = [j % len(base) for j in range(nc)]
    if c.sources is not None:
        s = dict(c.sources)
        for key in ("cqs", "csert"):
            s[key] = np.ascontiguousarray(np.asarray(s[key])[..., pick])
        c.sources = s
    if c.conc_bc is not None:
        b = dict(c.conc_bc)
        b["side"] = [None if d is None else
                     dict(d, cb=np.ascontiguousarray(np.asarray(d["cb"])[..., pick]),
                          csert=np.ascontiguousarray(np.asarray(d["csert"])[..., pick]))
                     for d in b["side"]]
        c.conc_bc = b
    return c


def _same(a, b, nc):
    for j in range(nc):
        x, x1 = a.get_constituent(j)
        y, y1 = b.get_constituent(j)
        assert np.array_equal(x, y) and np.array_equal(x1, y1), j


# a column kernel that takes the case (at most four waves, 64 KiB of LDS)
REF = {1: 1, 2: 2, 3: 1, 4: 1, 5: 2, 7: 2}


@pytest.mark.parametrize("store", ["fp64", "fp32"])
@pytest.mark.parametrize("kc,nc", [(1, 3), (2, 1), (3, 2), (7, 4), (8, 5), (15, 3), (21, 2),
                                   (41, 1), (9, 7)])
def test_layers_bitwise_column_kernels(kc, nc, store):
    from efdc_amd import grids, lib
    st = lib.STORE_FP64 if store == "fp64" else lib.STORE_FP32
    dz = np.linspace(1.0, 2.0, kc)
    case = _constituents(grids.tidal_basin(37, 19, kc, seed=60 + kc, dzck=dz), nc)
    a = _ctx(case, 0, store=st)
    b = _ctx(case, REF[nc], store=st)
    for n in range(1, 9):
        a.step(case.dt, n)
        b.step(case.dt, n)
    _same(a, b, nc)
    assert np.array_equal(a.get("P"), b.get("P"))
    a.close()
    b.close()


@pytest.mark.parametrize("store", ["fp64", "fp32"])
@pytest.mark.parametrize("kc", [43, 64])
def test_many_layers_in_fp64(kc, store):
    """One constituent on the largest columns that fit the LDS, against numpy
    (the oracle's column buffers end at 62 layers).  Bound: the storage's
    rounding per step (2^-24 relative in FP32) times the three steps and the
    few operations of a layer."""
    from efdc_amd import grids, lib
    st = lib.STORE_FP64 if store == "fp64" else lib.STORE_FP32
    case = _constituents(grids.transport_case(30, 17, kc, seed=5), 1)
    a = _ctx(case, 0, store=st)
    con = case.consts[0]["con"][:kc].copy()
    for n in (1, 2, 3):
        a.calconc(case.dt, n)
        con = _calconc_fp64(case, con)
    got = a.get_constituent(0)[0][:kc]
    tol = 1e-12 if store == "fp64" else 2e-6
    L = np.arange(2, case.grid.LA + 1) - 1
    assert np.max(np.abs(got[:, L] - con[:, L])) <= tol * np.max(np.abs(con))
    a.close()


def _calconc_fp64(case, con):
    """One CALCONC of a conservative constituent in numpy (closed basin)."""
    g, h, k, w, dt = case.grid, case.h, case.k, case.w, case.dt
    kc = g.KC
    m = {d: case.grid.maps[n] - 1 for d, n in dict(W="LWC", E="LEC", S="LSC", N="LNC").items()}
    u, v = k["UHDY2"][:kc], k["VHDX2"][:kc]
    fu = u * np.where(u >= 0, con[:, m["W"]], con)
    fv = v * np.where(v >= 0, con[:, m["S"]], con)
    wv = w["W2"][1:kc]
    fw = np.zeros((kc + 1, g.LCM))
    fw[1:kc] = wv * np.where(wv >= 0, con[:-1], con[1:])
    fq = np.zeros_like(con)
    s = case.sources
    for q, L in enumerate(s["LQS"]):
        fq[:, L - 1] += s["qss"][q] * s["cqs"][q, :, 0]
    new = (con * k["H1PK"][:kc] + dt * ((fq + fu - fu[:, m["E"]] + fv - fv[:, m["N"]]) *
                                        h["DXYIP"] + fw[:-1] - fw[1:])) * k["HPKI"][:kc]
    up = np.zeros_like(con)
    lo = np.zeros_like(con)
    up[:-1] = -dt * k["CDZKK"][:kc - 1] * h["HPI"] * k["AB"][:kc - 1]
    lo[1:] = -dt * k["CDZKMK"][1:kc] * h["HPI"] * k["AB"][:kc - 1]
    y, c = np.zeros_like(con), np.zeros_like(con)
    prev_y = prev_c = 0.0
    for q in range(kc):
        d = 1.0 - up[q] - lo[q] - lo[q] * prev_c
        y[q] = (new[q] - lo[q] * prev_y) / d
        c[q] = up[q] / d
        prev_y, prev_c = y[q], c[q]
    out = y.copy()
    for q in range(kc - 2, -1, -1):
        out[q] = y[q] - c[q] * out[q + 1]
    wet = np.zeros(g.LCM, bool)
    wet[1:g.LA] = True
    return np.where(wet, out, 0.0)


def test_layers_with_drying_and_without_the_solve():
    from efdc_amd import grids
    dry = _constituents(grids.drying_basin(40, 12, 3, seed=7), 3)
    a, b = _ctx(dry, 0, ISDRY=99), _ctx(dry, 1, ISDRY=99)
    for n in range(1, 13):
        a.step(dry.dt, n)
        b.step(dry.dt, n)
    assert (a.get_dry_state()[0][1:dry.grid.LA] == 0).any()
    _same(a, b, 3)
    a.close()
    b.close()
    # anti-diffusion: the column pass stops before the vertical solve
    adv = grids.transport_case(29, 23, 6, seed=9, isadac=1, isfct=1)
    a, b = _ctx(adv, 0), _ctx(adv, 1)
    for n in (1, 2, 3):
        a.calconc(adv.dt, n)
        b.calconc(adv.dt, n)
    _same(a, b, 4)
    a.close()
    b.close()
