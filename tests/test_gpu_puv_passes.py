"""The passes around the solve of CALPUV2C in the forms that depend on the
case: open-boundary rows in one workgroup or in launches of their own, tidal
constituents in the launch's arguments or in memory, a drying step whose plain
solve is repeated; FP64, against the oracle or the ordinary run."""
import numpy as np
import pytest

from conftest import eta_err, wet_index

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,mtide", [(6, 5, 1), (6, 1022, 16), (6, 1030, 17), (6, 40, 17),
                                         (6, 1300, 2), (520, 510, 1)])  # > 2**18 cells
def test_open_boundary_rows_and_tides(oracle_mod, nx, ny, mtide):
    from efdc_amd import grids
    from efdc_amd.lib import Context
    case = grids.tidal_basin(nx, ny, 2, seed=ny, amp=0.2)
    b = case.open_bc
    side = next(s for s in b["side"] if s is not None)
    n = len(side["pser"])
    rng = np.random.default_rng(mtide)
    b["mtide"] = mtide
    b["tcp"] = np.linspace(4000.0, 90000.0, mtide)
    for key in ("pcb", "psb"):
        side[key] = rng.normal(0.0, 2.0 / mtide, n * mtide).reshape(np.shape(side[key])[:0] + (-1,))
    ref = case.copy()
    o = oracle_mod.Oracle(ref, rsqm=1e-22, iterm=2000)
    ctx = Context(case.grid, RSQM=1e-22, ITERM=2000).upload_case(case)
    for k in range(1, 6):
        o.step(k)
        ctx.step(case.dt, k)
    L = wet_index(case)
    assert eta_err(ctx.get("P")[L], ref.h["P"][L]) <= 1e-9
    for name in ("HP", "HU", "HV", "HPI", "HUI", "HVI"):
        np.testing.assert_allclose(ctx.get(name)[L], ref.h[name][L], rtol=1e-9, err_msg=name)
    ctx.close()


@pytest.mark.parametrize("isdry", [1, 99])
def test_drying_step_repeats_an_abandoned_solve(isdry):
    from efdc_amd import grids
    from efdc_amd.lib import Context
    case = grids.drying_basin(120, 40, 2, seed=3)
    kw = dict(RSQM=1e-22, ITERM=2000, ISDRY=isdry)
    a = Context(case.grid, **kw).upload_case(case)
    b = Context(case.grid, **kw).upload_case(case)
    a.set_cg_launch(0, spin_limit=1)
    for k in range(1, 9):
        a.step(case.dt, k)
        b.step(case.dt, k)
    assert a.cg_launch()[1] >= 1 and b.cg_launch() == (0, 0)
    L = wet_index(case)
    np.testing.assert_array_equal(a.get_dry_state()[0], b.get_dry_state()[0])
    np.testing.assert_array_equal(a.get("SUB")[L], b.get("SUB")[L])
    assert eta_err(a.get("P")[L], b.get("P")[L]) <= 1e-9
    a.close()
    b.close()
