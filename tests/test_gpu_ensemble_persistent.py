"""The FP64 solve of an ensemble's basins in one persistent launch (the
default) against the two-launches-per-iteration solve: a basin's bits are its
own with either, whatever basins share the context, and the settings and
trials of the solve choose between them."""
import numpy as np
import pytest

from conftest import eta_err
from test_gpu_ensemble import _ctx, _tidal_ensemble

pytestmark = pytest.mark.gpu


def _many(n):
    from efdc_amd import grids
    return grids.concat_basins(
        [grids.tidal_basin(12 + 4 * (i % 4), 10 + 3 * (i % 2), 2, seed=300 + i,
                           amp=0.05 + 0.003 * (i % 50)) for i in range(n)])


def _lakes():
    from efdc_amd import grids
    return grids.concat_basins([grids.external_case(grids.lake_mask(n, n, s), seed=s)
                                for n, s in ((48, 31), (330, 32), (33, 33), (20, 35))])


# 5 basins; lakes of 100 to 50000 cells (several workgroups a basin); as many
# basins as workgroups of the chip; more than that (launch by launch)
@pytest.mark.parametrize("make,persistent", [
    (lambda: _tidal_ensemble()[1:], True), (_lakes, True),
    (lambda: _many(256), True), (lambda: _many(600), False),
])
def test_basins_persistent_against_launches(make, persistent):
    from efdc_amd import lib
    ens, first = make()
    a, b = _ctx(ens, cg_kernel=lib.CG_KERNEL_AUTO), _ctx(ens)
    for x in (a, b):
        x.set_segments(first)
    a.timers(True)
    for n in range(1, 7):
        a.calpuv2c(ens.dt, n)
        b.calpuv2c(ens.dt, n)
        ia, sa = a.segment_stats()
        ib, sb = b.segment_stats()
        assert not np.any(sa) and not np.any(sb)
        assert list(ia) == list(ib)
    assert ("cg_persistent64" in a.read_timers()) == persistent
    L = np.arange(1, ens.grid.LA)
    assert np.array_equal(a.get("P")[L], b.get("P")[L])
    a.close()
    b.close()


def test_basins_persistent_cap_and_repeated_launch():
    from efdc_amd import lib
    _, ens, first = _tidal_ensemble()
    c = _ctx(ens, cg_kernel=lib.CG_KERNEL_AUTO, RSQM=1e-30, ITERM=3)
    c.set_segments(first)
    with pytest.raises(lib.EfdcError) as e:
        c.calpuv2c(ens.dt, 1)
    assert e.value.status == 3
    it, status = c.segment_stats()
    assert list(it) == [3] * len(first) and list(status) == [3] * len(first)
    c.close()
    # a plain launch whose waits give up is repeated cooperatively
    a, b = _ctx(ens, cg_kernel=lib.CG_KERNEL_AUTO), _ctx(ens)
    a.set_segments(first)
    b.set_segments(first)
    a.set_cg_launch(0, spin_limit=1)
    a.calpuv2c(ens.dt, 1)
    b.calpuv2c(ens.dt, 1)
    assert a.cg_launch()[1] >= 1
    L = np.arange(1, ens.grid.LA)
    assert np.array_equal(a.get("P")[L], b.get("P")[L])
    a.close()
    b.close()


def _rect(nx, ny, seed):
    from efdc_amd import grids
    return grids.external_case(np.pad(np.ones((ny, nx), bool), 1), seed=seed, depth_sigma=2.0)


def _companies():
    """The same three basins (one tile, 11 tiles with a ragged end, 70 tiles) first,
    in the middle and last, beside small ones, beside one of 300 tiles and
    beside as many as leave two, four and six cells a thread."""
    from efdc_amd import grids
    three = [_rect(20, 17, 41),
             grids.external_case(grids.lake_mask(96, 88, 42), seed=42, depth_sigma=2.0),
             _rect(211, 169, 43)]
    small = [_rect(16 + i, 9 + i % 3, 50 + i) for i in range(4)]
    wide = [_rect(401, 383, 60)]
    many = [_rect(250, 201, 70 + i) for i in range(9)]
    return three, [(0, three + small), (4, small + three + wide), (9, many + three),
                   (1, wide + three + many)]


def test_basin_bits_do_not_depend_on_its_company():
    """With the kernel left to the library, which takes the persistent solve, a
    basin's fields are bit for bit those of the basin alone with
    CG_KERNEL_MULTI, whichever basins share its context; also where the launch
    was abandoned and repeated.  All basins of a context (up to 300 tiles, more
    than a reduction's 256 threads) against its solve by launches."""
    from efdc_amd import grids, lib
    fields = ["P", "P1", "HP", "H1P", "HU", "UHDYE", "VHDXE", "CCC", "CCS", "FPTMP"]
    three, companies = _companies()
    alone = []
    for b in three:
        c = _ctx(b)
        its = [c.calpuv2c(b.dt, n)["iters"] for n in (1, 2, 3)]
        alone.append((its, {f: c.get(f)[1:1 + b.grid.nwet] for f in fields}))
        c.close()
    for at, basins in companies:
        ens, first = grids.concat_basins(basins)
        m = _ctx(ens)
        m.set_segments(first)
        for n in (1, 2, 3):
            m.calpuv2c(ens.dt, n)
        for spin in (0, 1):
            c = _ctx(ens, cg_kernel=lib.CG_KERNEL_AUTO)
            c.set_segments(first)
            c.set_cg_launch(0, spin_limit=spin)
            c.timers(True)
            its = []
            for n in (1, 2, 3):
                c.calpuv2c(ens.dt, n)
                its.append(list(c.segment_stats()[0][at:at + 3]))
            assert "cg_persistent64" in c.read_timers()
            assert (c.cg_launch()[1] >= 1) == (spin == 1)
            for q in range(3):
                sl = grids.basin_slice(ens, first, at + q)
                assert [i[q] for i in its] == alone[q][0], (at, spin, q)
                for f in fields:
                    assert np.array_equal(c.get(f)[sl], alone[q][1][f]), (at, spin, q, f)
            for f in fields:
                assert np.array_equal(c.get(f)[1:ens.grid.LA], m.get(f)[1:ens.grid.LA]), (at, f)
            c.close()
        m.close()


def test_settings_of_the_basins_solve_act():
    """The tile and the replay of the per-basin launches select them; the
    trials time the persistent solve beside them and what they choose is what
    the next solve runs.  Every choice but another tile gives the same bits."""
    from efdc_amd import grids, lib
    ens, first = grids.concat_basins([_rect(120, 101, 5), _rect(64, 33, 6), _rect(90, 90, 7)])

    def run(setup, auto=True):
        kern = lib.CG_KERNEL_AUTO if auto else lib.CG_KERNEL_MULTI
        c = _ctx(ens, cg_kernel=kern)
        c.set_segments(first)
        setup(c)
        c.calpuv2c(ens.dt, 1)  # trials, if any
        c.timers(True)
        c.calpuv2c(ens.dt, 2)
        t = c.read_timers()
        p, rep, tile, rp = c.get("P"), c.tune_report(), c.segment_tile(), c.cg_replay()
        c.close()
        assert ("cg_persistent64" in t) != ("cg_spmv_pupdate" in t)
        return p, "cg_persistent64" in t, rep, tile, rp

    want = run(lambda c: None, auto=False)[0]
    for setup, persistent in ((lambda c: None, True), (lambda c: c.set_segment_tile(512), True),
                              (lambda c: c.set_cg_replay(1), False),
                              (lambda c: (c.set_cg_replay(1), c.set_cg_replay(0)), True)):
        p, pers, _, tile, _ = run(setup)
        assert pers == persistent and tile == 512
        assert np.array_equal(p, want)
    p, pers, _, tile, _ = run(lambda c: c.set_segment_tile(1024))
    assert not pers and tile == 1024
    assert eta_err(p, want) <= 1e-9
    for setup, names in (
            (lambda c: c.set_segment_tile(0), ["seg_cg_tile_256", "seg_cg_tile_512",
                                               "seg_cg_tile_1024", "seg_cg_tile_2048",
                                               "seg_cg_persistent"]),
            (lambda c: c.set_cg_replay(2), ["cg_fp64 launches", "cg_fp64 graphs",
                                            "cg_fp64 persistent"])):
        p, pers, rep, tile, rp = run(setup)
        assert list(rep["shapes"]) == names
        chosen = rep["chosen"]
        assert chosen == [min(names, key=rep["shapes"].get)]
        assert pers == chosen[0].endswith("persistent")
        assert rp == (1 if chosen[0].endswith("graphs") else 0)
        if chosen[0].startswith("seg_cg_tile_"):
            assert tile == int(chosen[0][12:])
        if tile == 512:
            assert np.array_equal(p, want)
