"""The transport autotuner: every launch shape it times gives the same bits,
and the choice persists for the following steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store", ["fp64", "fp32"])
def test_autotuned_transport_is_bitwise_the_default(store):
    from efdc_amd import grids, lib
    st = lib.STORE_FP64 if store == "fp64" else lib.STORE_FP32
    case = grids.tidal_basin(64, 32, 5, seed=8)
    a = lib.Context(case.grid, store=st).upload_case(case)
    b = lib.Context(case.grid, store=st).upload_case(case)
    a.autotune(True)
    for n in range(1, 6):
        a.step(case.dt, n)
        b.step(case.dt, n)
    rep = a.tune_report()
    print(rep)
    assert len(rep["shapes"]) >= 2 and len(rep["chosen"]) == 1
    assert rep["chosen"][0] in rep["shapes"]
    for j in range(len(case.consts)):
        ca, c1a = a.get_constituent(j)
        cb, c1b = b.get_constituent(j)
        assert np.array_equal(ca, cb) and np.array_equal(c1a, c1b)
    assert np.array_equal(a.get("P"), b.get("P"))
    a.close()
    b.close()


def test_autotuned_mixed_solve_degree():
    """With the mixed CG on the persistent solve, the tuner times the local
    preconditioner degrees from the same P, then the pipelined form at the
    fastest degree, keeps one, and the step's result stays within the
    mixed-precision bar of the FP64 solve."""
    from efdc_amd import grids, lib
    from conftest import eta_err, wet_index
    wet = grids.lake_mask(160, 160, 5)
    case = grids.external_case(wet, seed=5)
    m = lib.Context(case.grid, cg_mode=lib.CG_MIXED, RSQM=1e-20, ITERM=2000).upload_case(case)
    d = lib.Context(case.grid, cg_mode=lib.CG_FP64, RSQM=1e-24, ITERM=2000).upload_case(case)
    m.autotune(True)
    for n in (1, 2, 3):
        m.calpuv2c(case.dt, n)
        d.calpuv2c(case.dt, n)
    rep = m.tune_report()
    print(rep)
    degs = [k for k in rep["shapes"] if k.startswith("pcg_mixed degree=")]
    forms = [k for k in rep["shapes"] if k.startswith("pcg_mixed pipelined")]
    assert len(degs) == 5 and len(forms) == 1
    assert len([k for k in rep["chosen"] if k.startswith("pcg_mixed")]) == 1
    assert m.cg_pipeline() == (2 if forms[0] in rep["chosen"] else 1)
    i = wet_index(case)
    assert eta_err(m.get("P")[i], d.get("P")[i]) <= 1e-6
    m.close()
    d.close()


@pytest.mark.parametrize("kc", [5, 64])
def test_constituent_added_after_tuning(kc):
    """A constituent that is added after the tuner has chosen a column kernel
    may leave no column shape that fits (64 layers in FP64: one fills the
    64 KiB, two take 96): the next step runs a kernel that fits, with the bits
    of a context that was never tuned."""
    from efdc_amd import grids, lib
    case = grids.tidal_basin(130, 120, kc, seed=8)
    case.sources = case.conc_bc = case.open_bc = None
    both = case.consts
    one, two = case.copy(), case.copy()
    one.consts = [both[0]]
    a = lib.Context(one.grid).upload_case(one)
    a.autotune(True)
    for n in (1, 2):
        a.calconc(case.dt, n)
    assert len(a.tune_report()["chosen"]) == 1
    con, con1 = a.get_constituent(0)
    c = both[1]
    slot = a.add_constituent(c["mo"], c["isadac"], c["isfct"], c["rkdye"], c["is_dye"])
    a.set_constituent(slot, c["con"], c["con1"])
    two.consts = [dict(both[0], con=con, con1=con1), dict(c, wset=0.0)]
    b = lib.Context(two.grid).upload_case(two)
    for n in (3, 4):
        a.calconc(case.dt, n)
        b.calconc(case.dt, n)
    for j in range(2):
        assert all(np.array_equal(x, y) for x, y in zip(a.get_constituent(j),
                                                        b.get_constituent(j))), j
    a.close()
    b.close()


def test_column_kernels_are_timed_with_their_settling():
    """The layer kernel settles in its own pass, the column kernels need a
    launch for it: the tuner times both with the settling, and the step it
    tunes on gives the bits of an untuned one."""
    from efdc_amd import grids, lib
    case = grids.tidal_basin(64, 48, 6, seed=8)
    case.consts[1].update(wset=3e-4, probdep=0.6, wese=1e-6)
    a = lib.Context(case.grid).upload_case(case)
    b = lib.Context(case.grid).upload_case(case)
    a.timers(True)
    a.autotune(True)
    a.calconc(case.dt, 1)
    b.calconc(case.dt, 1)
    rep = a.tune_report()
    columns = [n for n in rep["shapes"] if n.startswith("tran_colm")]
    assert "tran_layers" in rep["shapes"] and columns
    n = a.read_timers()["settle"][0]
    assert n == 4 * len(columns) + (rep["chosen"][0] != "tran_layers")
    a.calconc(case.dt, 2)
    b.calconc(case.dt, 2)
    for j in range(len(case.consts)):
        assert all(np.array_equal(x, y) for x, y in zip(a.get_constituent(j),
                                                        b.get_constituent(j))), j
    a.close()
    b.close()
