"""The multigrid legs that run a level's sweeps in one launch, against the
oracle's V-cycle sweep by sweep: grids at the edges of the blocks (64 columns,
24 and 32 rows, two-plane chunks), smaller than the overlap, odd and periodic,
with two and three sweeps (and four, which run one by one but in the small
levels), in FP64 and with the FP32 finest levels.  Solves
stopped after two iterations, so that x holds two V-cycles and no limit."""
import numpy as np
import pytest

from cajitafluids_amd import configs as K
from helpers import gpu_to_oracle, rel_l2

pytestmark = pytest.mark.gpu

GRIDS = [
    ((3, 3, 3), (1, 1, 1)), ((5, 4, 3), (0, 0, 0)), ((64, 32, 6), (0, 0, 0)),
    ((65, 33, 7), (0, 0, 1)), ((58, 26, 9), (1, 1, 0)), ((59, 27, 12), (1, 1, 1)),
    ((122, 57, 5), (0, 1, 0)), ((130, 60, 18), (0, 0, 0)), ((96, 80, 72), (1, 0, 0)),
    ((64, 24, 1), (0, 0, 0)), ((65, 33, 1), (0, 1, 0)), ((3, 4, 1), (1, 0, 0)),
    ((187, 121, 1), (1, 1, 0)),
]


@pytest.mark.parametrize("precision", [K.FP64, K.FP32_REFINED])
@pytest.mark.parametrize("nu", [2, 3, 4])
@pytest.mark.parametrize("n,periodic", GRIDS)
def test_mg_legs(oracle_mod, n, periodic, nu, precision):
    dim = 3 if n[2] > 1 else 2
    if dim == 2 and precision != K.FP64:
        pytest.skip("FP32 levels are 3-D")
    check_solve(oracle_mod, n, periodic, nu, precision)


# levels whose legs run in blocks of 16 and of 12 waves: level 0, and levels 0
# (padded) and 1 (boxes)
@pytest.mark.parametrize("n,periodic", [((130, 121, 96), (0, 1, 0)), ((247, 243, 159), (0, 0, 0))])
def test_mg_legs_large(oracle_mod, n, periodic):
    check_solve(oracle_mod, n, periodic, 3, K.FP64)


def check_solve(oracle_mod, n, periodic, nu, precision):
    from cajitafluids_amd import _lib
    from cajitafluids_amd.solver import Solver
    dim = 3 if n[2] > 1 else 2
    cfg = K.base_config(dim, n[0])
    cfg.update(num_cell=list(n), hi=[1.0, n[1] / n[0], n[2] / n[0] if dim == 3 else 1.0],
               clamp_dt=0, dt=0.002, halo=1, field_order=1, periodic=list(periodic),
               preconditioner=K.PRECOND_MG, precision=precision, mg_nu=nu, cg_max_iter=2,
               cg_tol=1e-30)
    cfg["wall_type"][dim - 1][1] = K.FREE
    print(f"mg legs: {n} {periodic} nu {nu} precision {precision}", flush=True)
    sol, orc = Solver(cfg), oracle_mod.Oracle(cfg)
    sol.init_random_faces(5)
    gpu_to_oracle(sol, orc)
    for o in (sol, orc):
        o.build_rhs()
        o.rhs_remove_mean()
    with pytest.raises(_lib.CfError) as ei:
        sol.pressure_solve(precision)
    assert ei.value.code == _lib.CF_ENOCONV
    rc, _ = orc.pressure_solve(precision)
    assert rc == _lib.CF_ENOCONV
    x_g = sol.owned_view(sol.get_pressure(0), 0)
    x_o = orc.owned_view(orc.lhs(), 0)
    assert np.any(x_o != 0.0)
    assert rel_l2(x_g, x_o) <= 1e-12
    sol.close()
    orc.close()
