"""The cooperative 3-D solve (a workgroup per pencil of x-rows): pencil shapes
with one to four partials a lane of the gather, ragged last pencils, axes of
one to three cells, periodic axes inside and across pencils; x bit for bit the
oracle's after an odd and an even number of iterations, and across two
launches."""
import numpy as np
import pytest

from cajitafluids_amd import configs as K
from helpers import gpu_to_oracle

pytestmark = pytest.mark.gpu

GRIDS = [
    ((3, 2, 1), (0, 0, 0)), ((4, 4, 4), (1, 1, 1)), ((7, 1, 9), (0, 0, 1)),
    ((12, 12, 12), (0, 0, 0)), ((33, 17, 9), (1, 0, 0)), ((20, 31, 40), (0, 1, 1)),
    ((45, 52, 61), (0, 0, 0)), ((64, 64, 64), (1, 1, 0)), ((90, 70, 81), (0, 0, 0)),
    ((130, 40, 30), (0, 1, 0)),
]


@pytest.mark.parametrize("precond", [K.PRECOND_JACOBI, K.PRECOND_NONE])
@pytest.mark.parametrize("n,periodic", GRIDS)
@pytest.mark.parametrize("maxit", [1, 4, 259])
def test_coop_pencils(oracle_mod, n, periodic, maxit, precond):
    from cajitafluids_amd import _lib
    from cajitafluids_amd.solver import Solver
    if maxit > 4 and n[0] * n[1] * n[2] > 30000:
        pytest.skip("two launches: on the smaller grids")
    cfg = K.base_config(3, n[0])
    cfg.update(num_cell=list(n), hi=[1.0, n[1] / n[0], n[2] / n[0]], clamp_dt=0, dt=0.002,
               halo=1, field_order=1, periodic=list(periodic), cg_max_iter=maxit, cg_tol=1e-300,
               preconditioner=precond)
    cfg["wall_type"][1][0] = K.FREE
    print(f"coop pencils: {n} {periodic} maxit {maxit} precond {precond}", flush=True)
    sol, orc = Solver(cfg), oracle_mod.Oracle(cfg)
    sol.set_kernel_timing(True)
    sol.init_random_faces(5)
    gpu_to_oracle(sol, orc)
    for o in (sol, orc):
        o.build_rhs()
        o.rhs_remove_mean()
    for _ in range(2):  # the second solve's exchanges follow the first's
        try:
            sol.pressure_solve(K.FP64)
            code = 0
        except _lib.CfError as e:
            code = e.code
    rc, st_o = orc.pressure_solve(K.FP64)
    assert code == rc
    assert sol.last_stats["iterations"] == st_o["iterations"]
    assert sol.kernel_time(_lib.TK_PCG_COOP)[1] >= 2
    assert sol.kernel_time(_lib.TK_DIR_SPMV)[1] == 0
    x_g = sol.owned_view(sol.get_pressure(0), 0)
    x_o = orc.owned_view(orc.lhs(), 0)
    assert np.any(x_o != 0.0)
    assert np.array_equal(x_g, x_o)
    sol.close()
    orc.close()
