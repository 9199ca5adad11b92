"""The streaming tile kernels of the 3-D PCG against the oracle, x bit for bit,
on grids whose rows (more than 1024 cells) the cooperative solve refuses:
solves stopped after odd and even counts (an update leaves x alone on every
second iteration), with and without the Jacobi preconditioner, in FP64 and as
one FP32 pass; and refined solves that carry the direction over passes of odd
and of even length (the next pass starts on the x and the direction that the
last one left)."""
import numpy as np
import pytest

from cajitafluids_amd import configs as K

pytestmark = pytest.mark.gpu

# partial tiles along every axis, chunks that end in one plane, periodic axes
GRIDS = [((1030, 17, 9), (0, 0, 0)), ((1027, 20, 35), (1, 0, 1)), ((1089, 33, 5), (0, 1, 0))]


def _pair(oracle_mod, n, periodic, **kw):
    from cajitafluids_amd.solver import Solver
    cfg = K.base_config(3, n[0])
    cfg.update(num_cell=list(n), hi=[1.0, n[1] / n[0], n[2] / n[0]], clamp_dt=0, dt=0.002,
               halo=1, field_order=1, periodic=list(periodic), **kw)
    cfg["wall_type"][0][1] = K.FREE
    sol, orc = Solver(cfg), oracle_mod.Oracle(cfg)
    sol.set_kernel_timing(True)
    rng = np.random.default_rng(11)
    for e in range(1, 4):
        f = sol.get(e)
        own = sol.owned_view(f, e)
        own[...] = rng.standard_normal(own.shape)
        sol.set(e, f)
        orc.field(e)[...] = f
    for o in (sol, orc):
        o.build_rhs()
        o.rhs_remove_mean()
    return sol, orc


def _solve(sol, orc, precision, timed):
    """Both solves: equal counts and status, x bit for bit, by the tiles."""
    from cajitafluids_amd import _lib
    try:
        sol.pressure_solve(precision)
        code = 0
    except _lib.CfError as e:
        code = e.code
    rc, st = orc.pressure_solve(precision)
    assert code == rc
    assert sol.last_stats["iterations"] == st["iterations"]
    assert sol.last_stats["outer_iterations"] == st["outer_iterations"]
    assert sol.kernel_time(timed)[1] >= st["iterations"]
    assert sol.kernel_time(_lib.TK_PCG_COOP)[1] == 0
    x_g = sol.owned_view(sol.get_pressure(0), 0)
    x_o = orc.owned_view(orc.lhs(), 0)
    assert np.any(x_o != 0.0)
    assert np.array_equal(x_g, x_o)
    sol.close()
    orc.close()
    return st["iterations"]


@pytest.mark.parametrize("precision", [K.FP64, K.FP32_REFINED])
@pytest.mark.parametrize("precond", [K.PRECOND_JACOBI, K.PRECOND_NONE])
@pytest.mark.parametrize("maxit", [1, 2, 5, 6])
@pytest.mark.parametrize("n,periodic", GRIDS)
def test_tiles_truncated(oracle_mod, n, periodic, maxit, precond, precision):
    from cajitafluids_amd import _lib
    print(f"pcg tiles: {n} {periodic} maxit {maxit} precond {precond} precision {precision}",
          flush=True)
    sol, orc = _pair(oracle_mod, n, periodic, precision=precision, preconditioner=precond,
                     cg_max_iter=maxit, cg_tol=1e-30, refine_mode=K.REFINE_RESTART,
                     inner_max_iter=0)
    timed = _lib.TK_DIR_SPMV if precision == K.FP64 else _lib.TK_DIR_SPMV32
    assert _solve(sol, orc, precision, timed) == maxit


# a pass's inner tolerance, and the passes' lengths on the three grids: odd and
# even ones follow each other in every order
CARRY = [(0.5, [[1, 1, 2, 4], [1, 1, 2, 3], [1, 1, 2, 4]]),
         (0.3, [[2, 4], [2, 3, 7, 58], [2, 4]]),
         (0.1, [[3, 137], [3, 13], [4, 287]])]


@pytest.mark.parametrize("itol,lengths", [(t, z) for t, ls in CARRY for z in zip(GRIDS, ls)])
def test_tiles_carry(oracle_mod, itol, lengths):
    from cajitafluids_amd import _lib
    (n, periodic), passes = lengths
    print(f"pcg tiles carry: {n} {periodic} inner_tol {itol} passes {passes}", flush=True)
    sol, orc = _pair(oracle_mod, n, periodic, precision=K.FP32_REFINED, cg_tol=1e-14,
                     refine_mode=K.REFINE_CARRY, inner_tol=itol, max_outer=len(passes))
    assert _solve(sol, orc, K.FP32_REFINED, _lib.TK_DIR_SPMV32) == sum(passes)


@pytest.mark.parametrize("n,periodic", GRIDS)
def test_tiles_carry_unpreconditioned(oracle_mod, n, periodic):
    from cajitafluids_amd import _lib
    print(f"pcg tiles carry: {n} {periodic} unpreconditioned", flush=True)
    sol, orc = _pair(oracle_mod, n, periodic, precision=K.FP32_REFINED, cg_tol=1e-14,
                     preconditioner=K.PRECOND_NONE, refine_mode=K.REFINE_CARRY, inner_tol=0.5,
                     max_outer=4)
    assert _solve(sol, orc, K.FP32_REFINED, _lib.TK_DIR_SPMV32) in (7, 8)
