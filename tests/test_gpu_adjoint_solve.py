"""The adjoint's solve, seeds and gather: gradients of a short window with the
persistent solve (the default) against the launch-by-launch one, and a seed
list longer than one chunk with repeated entries against the sequential sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,kc", [(9, 7, 1), (31, 22, 3), (65, 40, 13)])
def test_gradient_persistent_against_launches(nx, ny, kc):
    from efdc_amd import adjoint, grids, lib
    out = []
    for kernel in (lib.CG_KERNEL_AUTO, lib.CG_KERNEL_MULTI):
        case = grids.tidal_basin(nx, ny, kc, seed=4, amp=0.1)
        obs = np.arange(2, case.grid.LA + 1)[:: max(1, case.grid.LA // 7)]
        data = np.zeros((2, len(obs)))
        prob = adjoint.DyeMisfit(case, nsteps=4, obs_L=obs, obs_every=2, data=data, ckpt=2,
                                 store=lib.STORE_FP64, cg_kernel=kernel)
        loads = np.full((4, prob.nsrc), 2.0)
        out.append(prob.gradient(loads)[:3])
        prob.close()
    (J0, g0, n0), (J1, g1, n1) = out
    # the two solves stop at 1e-12 of the right-hand side
    assert abs(J0 - J1) <= 1e-9 * abs(J1)
    assert np.max(np.abs(g0 - g1)) <= 1e-8 * np.max(np.abs(g1))
    assert np.max(np.abs(n0 - n1)) <= 1e-8 * np.max(np.abs(n1))


@pytest.mark.parametrize("n", [1, 512, 513, 1700])
def test_seed_list_repeated_entries(n):
    from efdc_amd import adjoint, grids, lib
    case = grids.tidal_basin(14, 9, 3, seed=6, amp=0.1)
    prob = adjoint.DyeMisfit(case, nsteps=2, obs_L=np.array([5, 9]), obs_every=2,
                             data=np.zeros((1, 2)), ckpt=2, store=lib.STORE_FP64)
    rng = np.random.default_rng(n)
    L = rng.integers(2, case.grid.LA + 1, n)
    K = rng.integers(1, 4, n)
    v = rng.normal(size=n) * 10.0 ** rng.integers(-8, 8, n)
    want = np.zeros((3, case.grid.LCM))
    for a, b, x in zip(L, K, v):
        want[b - 1, a - 1] += x
    prob.ctx.adj_reset()
    prob.ctx.adj_seed_con(prob.dye, L, K, v)
    got = prob.ctx.adj_get(lib.ADJ_CON + prob.dye)
    np.testing.assert_array_equal(got[:3], want)
    prob.close()
