"""Anti-diffusion passes of several constituents at a time: more of them than
one group holds, with and without the limiter or the passes, at layer counts
around the finishing kernel's waves and at a ragged last tile, FP64, against
the oracle bit for bit."""
import numpy as np
import pytest

from test_gpu_tran_layers import _constituents

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kc,nx,ny,nconst", [
    (1, 13, 9, 2), (2, 63, 1, 3), (4, 17, 9, 9), (5, 11, 29, 12), (13, 23, 7, 4),
    (64, 9, 8, 2),
])
def test_adac_groups_bitexact(oracle_mod, kc, nx, ny, nconst):
    from efdc_amd import grids
    from efdc_amd.lib import Context
    case = _constituents(grids.transport_case(nx, ny, kc, seed=kc, isadac=1, isfct=0), nconst)
    for j, c in enumerate(case.consts):
        c["isadac"] = 0 if j % 4 == 2 else 1
        c["isfct"] = 1 if kc > 1 and j % 3 == 0 else 0
    ref = case.copy()
    o = oracle_mod.Oracle(ref)
    ctx = Context(case.grid).upload_case(case)
    for n in (1, 2, 3):
        o.calconc(niter=n)
        ctx.calconc(case.dt, n)
        for j, c in enumerate(ref.consts):
            con, con1 = ctx.get_constituent(j)
            np.testing.assert_array_equal(con[:kc], c["con"][:kc], err_msg=f"CON {j} n={n}")
            np.testing.assert_array_equal(con1[:kc], c["con1"][:kc], err_msg=f"CON1 {j} n={n}")
    ctx.close()
