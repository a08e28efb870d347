"""The two forms of CALUVW's column step (a thread per column; the layers of
a column side by side):

* at the edges of the rule that chooses between them, one call against the
  oracle from the same state, FP64, bit for bit;
* against each other, bit for bit in FP64 and FP32 storage, at every layer
  count with a column instance of its own: a small basin alone (layers) and
  beside one large enough that the grid takes the columns;
* drying and rewetting steps against the oracle with each of them.
"""
import numpy as np
import pytest

from conftest import wet_index
from edge_cases import edge_basin
from test_gpu_uvw import H_OUT, K_OUT, W_OUT, _compare_steps, _ready_for_caluvw

pytestmark = pytest.mark.gpu

G = 9.81


def _basin(kc, nx, ny):
    """Closed basin with a tilted surface and the internal mode's arrays."""
    from efdc_amd import grids
    case = grids.tidal_basin(nx, ny, kc, seed=kc, dt=5.0)
    case.open_bc = None
    case.conc_bc = None
    g, h, k = case.grid, case.h, case.k
    L = wet_index(case)
    eta = 0.2 * np.cos(np.pi * g.IL[L] / nx) + 0.1 * np.cos(np.pi * g.JL[L] / ny)
    h["HP"][L] = -h["BELV"][L] + eta
    h["H1P"][:] = h["HP"]
    h["H2P"][:] = h["HP"]
    h["P"][L] = G * eta
    h["P1"][:] = h["P"]
    grids.update_depth_arrays(g, h)
    grids.layer_depths(g, h, k)
    k["H1PK"][:] = k["HPK"]
    grids.add_internal_mode(case, av=1e-2)
    return case


@pytest.mark.parametrize("kc,nx,ny", [
    (2, 9, 7), (3, 17, 8),      # columns: too few layers for a wave each
    (4, 21, 3), (9, 33, 31),    # layers: a full tile and no more, a ragged last one
    (64, 10, 8),                # columns: more LDS than a CU has
    (5, 190, 190),              # columns: 565 tiles
    (6, 222, 221),              # layers: 767 tiles, the most
    (6, 222, 222),              # columns: 771 tiles
    (9, 190, 190),              # layers: a count without straight-line columns
    (12, 257, 256),             # layers: 1029 tiles
])
def test_caluvw_layer_and_column_kernels(oracle_mod, kc, nx, ny):
    from efdc_amd.lib import Context
    case = _basin(kc, nx, ny)
    o = _ready_for_caluvw(case, oracle_mod, nsteps=1)
    snap = case.copy()
    ctx = Context(snap.grid, RSQM=1e-26, ITERM=3000).upload_case(snap)
    assert o.caluvw() == 0
    ctx.caluvw(case.dt, 2)
    L = wet_index(case)
    for names, src, n in ((K_OUT, case.k, kc), (W_OUT, case.w, kc + 1)):
        for name in names:
            np.testing.assert_array_equal(ctx.get(name)[:n, L], src[name][:n, L], err_msg=name)
    for name in H_OUT:
        np.testing.assert_array_equal(ctx.get(name)[L], case.h[name][L], err_msg=name)
    ctx.close()


def _open_basin(kc, nx, ny, seed):
    """edge_basin (open on all four sides) with the internal mode's arrays and
    wind stresses."""
    from efdc_amd import grids
    case = grids.add_internal_mode(edge_basin(seed, nx=nx, ny=ny, kc=kc), av=5e-3)
    L = wet_index(case)
    rng = np.random.default_rng(seed)
    for key in ("TSX", "TSY"):
        case.h[key][L] = rng.normal(0, 1e-4, len(L))
    return case


@pytest.mark.parametrize("shear", [0, 1])
@pytest.mark.parametrize("kc", [4, 5, 6, 8, 10, 12, 16, 20])
def test_layers_equal_columns(oracle_mod, kc, shear):
    from efdc_amd import grids
    from efdc_amd.lib import STORE_FP32, STORE_FP64, Context
    case = _open_basin(kc, 23, 13, 40 + kc)
    _ready_for_caluvw(case, oracle_mod, nsteps=3, wind=1)
    if shear == 0:  # the shears and viscosities as the host set them
        rng = np.random.default_rng(kc)
        L = wet_index(case)
        for key in ("DU", "DV"):
            case.k[key][:kc - 1, L] = rng.uniform(-1e-6, 1e-6, (kc - 1, len(L)))
        for key in ("AVUI", "AVVI"):
            case.k[key][:kc - 1, L] = rng.uniform(50.0, 2000.0, (kc - 1, len(L)))
    large = _open_basin(kc, 226, 222, 3)
    large.conc_bc["wtci"] = case.conc_bc["wtci"]  # (concat_basins wants them shared)
    both, _ = grids.concat_basins([case, large])
    n = case.grid.nwet
    assert n <= 512 * 64 and 768 * 64 < both.grid.nwet <= 1024 * 64 - 64
    for store in (STORE_FP64, STORE_FP32):
        out = []
        for c in (case, both):
            ctx = Context(c.grid, RSQM=1e-26, ITERM=3000, store=store).upload_case(c)
            ctx.caluvw(c.dt, 4, shear=shear, wind=1)
            out.append({x: np.atleast_2d(ctx.get(x))[:, 1:n + 1] for x in K_OUT + W_OUT + H_OUT})
            ctx.close()
        for x in out[0]:
            np.testing.assert_array_equal(out[0][x], out[1][x], err_msg=f"{x} store {store}")


@pytest.mark.parametrize("store,tol_eta,tol_rel", [(0, 1e-9, 1e-9), (1, 1e-6, 1e-5)])
@pytest.mark.parametrize("nx,ny,kc,nsteps", [
    (40, 12, 5, 60),     # layers
    (320, 180, 4, 16),   # columns: 901 tiles
    (40, 12, 9, 30),     # layers: a count without straight-line columns
])
def test_drying_steps_layers_and_columns(oracle_mod, nx, ny, kc, nsteps, store, tol_eta, tol_rel):
    """Dry columns zeroed, faces beside them, the averages over them."""
    from efdc_amd import grids
    case = grids.add_internal_mode(grids.drying_basin(nx, ny, kc, deep=2.0), av=5e-3)
    _compare_steps(case, oracle_mod, nsteps, tol_eta, tol_rel, store=store, isdry=99, hdry=0.2)
