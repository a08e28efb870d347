"""The two forms of CALUVW's column step (a thread per column; the layers of
a column side by side) at the edges of the rule that chooses between them,
one call against the oracle from the same state, FP64, bit for bit."""
import numpy as np
import pytest

from conftest import wet_index
from test_gpu_uvw import H_OUT, K_OUT, W_OUT, _ready_for_caluvw

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
