"""The adjoint's solve, seeds and gather: gradients of a short window with the
persistent solve (the default) against the launch-by-launch one, also where
every plain launch gives up and its solve is repeated, and a seed list longer than one chunk with repeated entries against the sequential sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(nx, ny, kc, kernel):
    """Four steps of a basin whose dye varies from cell to cell and is observed
    in a seventh of the cells at every second step, so that the misfit depends on the
    transports and every step's adjoint system has a right-hand side."""
    from efdc_amd import adjoint, grids, lib
    case = grids.tidal_basin(nx, ny, kc, seed=4, amp=0.1)
    L = np.arange(2, case.grid.LA + 1) - 1
    rng = np.random.default_rng(nx)
    con = np.zeros_like(case.consts[1]["con"])
    con[:kc, L] = rng.uniform(1.0, 2.0, (kc, len(L)))
    case.consts[1].update(con=con, con1=con.copy())
    obs = np.arange(2, case.grid.LA + 1)[:: 7]
    return adjoint.DyeMisfit(case, nsteps=4, obs_L=obs, obs_every=2,
                             data=np.zeros((2, len(obs))), ckpt=2, store=lib.STORE_FP64,
                             cg_kernel=kernel)


def _close(a, b):
    # both solves stop at 1e-12 of the right-hand side
    (J0, g0, n0), (J1, g1, n1) = a, b
    assert J0 > 0.0 and np.max(np.abs(g0)) > 0.0 and np.max(np.abs(n0)) > 0.0
    assert abs(J0 - J1) <= 1e-9 * abs(J1)
    assert np.max(np.abs(g0 - g1)) <= 1e-8 * np.max(np.abs(g1))
    assert np.max(np.abs(n0 - n1)) <= 1e-8 * np.max(np.abs(n1))


@pytest.mark.parametrize("nx,ny,kc", [(9, 7, 1), (31, 22, 3), (65, 40, 13)])
def test_gradient_persistent_against_launches(nx, ny, kc):
    from efdc_amd import lib
    out = []
    for kernel in (lib.CG_KERNEL_AUTO, lib.CG_KERNEL_MULTI):
        prob = _problem(nx, ny, kc, kernel)
        prob.ctx.timers(True)
        *grad, stats = prob.gradient(np.full((4, prob.nsrc), 2.0))
        its = stats["adj_cg_iters"]
        assert len(its) == 4 and min(its) > 1
        # one launch a solve, or one and two an iteration
        n = prob.ctx.read_timers()["adj_cg"][0]
        assert n == 4 if kernel == lib.CG_KERNEL_AUTO else n >= 4 + 2 * sum(its)
        out.append(grad)
        prob.close()
    _close(*out)


def test_gradient_with_abandoned_launches():
    """Plain launches whose waits give up at once: the recorded steps' solves
    (repeated with the passes and the recording behind them) and the adjoint's
    own are solved again, and the gradient is the ordinary one."""
    from efdc_amd import lib
    out = []
    for spin in (0, 1):
        prob = _problem(95, 80, 3, lib.CG_KERNEL_AUTO)
        prob.ctx.set_cg_launch(0, spin_limit=spin)
        prob.ctx.timers(True)
        out.append(prob.gradient(np.full((4, prob.nsrc), 2.0))[:3])
        adj = prob.ctx.read_timers()["adj_cg"][0] - 4  # (4 adjoint solves)
        forward = prob.ctx.cg_launch()[1] - adj
        print("repeated solves: forward", forward, "adjoint", adj)
        assert (forward >= 4 and adj >= 2) if spin else (forward == 0 and adj == 0)
        prob.close()
    _close(*out)


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
