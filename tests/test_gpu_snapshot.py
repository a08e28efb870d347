"""State snapshots (efdc_state_save, efdc_state_load): the one-launch copy of
an aligned device buffer against the piece-by-piece copies that any other
buffer takes, on arrays whose bytes are no multiple of 16, and both
directions against the arrays themselves."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, kc, internal): snapshots below and above 64 MiB, odd and even LCM,
# with and without the internal mode's pieces (more than one launch's table)
SIZES = [(3, 3, 1, False), (16, 8, 3, False), (37, 23, 5, True), (331, 293, 11, False)]


class _DeviceBytes:
    """n device bytes set to 0xAB, from the HIP runtime that the library runs
    on (torch brings a runtime of its own, which finds no device once the
    library's is in use)."""

    def __init__(self, n):
        with open("/proc/self/maps") as f:
            paths = [ln.split()[-1] for ln in f if "libamdhip64.so" in ln]
        path = next((q for q in paths if "/torch/" not in q), paths[0])
        self.hip, self.n, self.p = C.CDLL(path), n, C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.p), C.c_size_t(n)) == 0
        h = np.full(n, 0xAB, np.uint8)
        assert self.hip.hipMemcpy(self.p, C.c_void_p(h.ctypes.data), C.c_size_t(n), 1) == 0

    def get(self):
        h = np.empty(self.n, np.uint8)
        assert self.hip.hipMemcpy(C.c_void_p(h.ctypes.data), self.p, C.c_size_t(self.n), 2) == 0
        return h

    def free(self):
        assert self.hip.hipFree(self.p) == 0


@pytest.mark.parametrize("store", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,kc,internal", SIZES)
def test_snapshot_copies(nx, ny, kc, internal, store):
    from efdc_amd import grids, lib
    case = grids.tidal_basin(nx, ny, kc, seed=nx)
    if internal:
        grids.add_internal_mode(case, av=1e-3)
    st = lib.STORE_FP32 if store == "fp32" else lib.STORE_FP64
    ctx = lib.Context(case.grid, store=st, RSQM=1e-20, ITERM=500)
    ctx.upload_case(case)
    for n in (1, 2):
        ctx.step(case.dt, n, internal=internal)
    names = ["P", "HP", "H2P", "UHDYE", "CCCI", "SVBO", "HPK", "UHDY2", "W2"]
    names += ["U1", "AVVI", "W"] if internal else []
    want = {a: ctx.get(a) for a in names}
    cons = [ctx.get_constituent(j) for j in range(2)]
    nb = ctx.state_bytes()
    # 0xAB in the gaps between the pieces, which no copy may touch
    a, b = _DeviceBytes(nb), _DeviceBytes(nb + 8)
    ctx.state_save(a.p.value)
    ctx.state_save(b.p.value + 8)
    ctx.synchronize()
    np.testing.assert_array_equal(a.get(), b.get()[8:])
    other = lib.Context(case.grid, store=st, RSQM=1e-20, ITERM=500)
    other.upload_case(case)
    if internal:
        other.step(case.dt, 1, internal=True)
    for buf in (a.p.value, b.p.value + 8):
        for name in ("P", "HPK", "W2"):
            other.set(name, np.ones_like(want[name]))
        other.state_load(buf)
        for name in names:
            assert np.array_equal(other.get(name), want[name]), name
        for j in range(2):
            got = other.get_constituent(j)
            assert np.array_equal(got[0], cons[j][0]) and np.array_equal(got[1], cons[j][1])
    ctx.close()
    other.close()
    a.free()
    b.free()


@pytest.mark.parametrize("align", [0, 8])
def test_short_buffer_is_refused(align):
    """A device buffer that ends within the snapshot is refused on the host
    before anything is copied, in both directions, also where the one-launch
    copy would take it (16-byte aligned)."""
    from efdc_amd import grids, lib
    case = grids.tidal_basin(100, 80, 2, seed=9)
    ctx = lib.Context(case.grid, RSQM=1e-20, ITERM=500)
    ctx.upload_case(case)
    ctx.step(case.dt, 1)
    nb = ctx.state_bytes()
    p = ctx.get("P")
    whole, short = _DeviceBytes(nb + 8), _DeviceBytes(nb // 2)
    for call in (ctx.state_save, ctx.state_load):
        with pytest.raises(lib.EfdcError) as e:
            call(short.p.value + align)
        assert e.value.status == 1
    assert np.all(short.get() == 0xAB)
    assert np.array_equal(ctx.get("P"), p)
    ctx.state_save(whole.p.value + align)
    ctx.step(case.dt, 2)
    ctx.state_load(whole.p.value + align)
    assert np.array_equal(ctx.get("P"), p)
    ctx.close()
    whole.free()
    short.free()
