"""The z chunks of the 3-D PCG tiles: grids whose chunks are one, two or
three planes deep, end in a shorter chunk, or fill the GPU unevenly, against
the oracle bit for bit (truncated solves: every iterate, not the limit).
Grids of up to about 100^3 with rows of at most 1024 cells run cooperatively;
the longer rows and the largest grid run the tiles."""
import numpy as np
import pytest

from cajitafluids_amd import configs as K
from helpers import gpu_to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [K.FP64, K.FP32_REFINED])
@pytest.mark.parametrize("n,periodic", [
    ((7, 5, 1), (0, 0, 0)), ((9, 6, 2), (0, 0, 0)), ((33, 17, 3), (1, 0, 0)),
    ((65, 15, 7), (0, 1, 1)), ((45, 52, 61), (0, 0, 0)), ((129, 33, 10), (1, 1, 0)),
    ((150, 141, 83), (0, 0, 1)), ((1025, 5, 1), (0, 0, 0)), ((1030, 17, 2), (1, 0, 0)),
    ((1100, 15, 7), (0, 1, 1)), ((1026, 33, 20), (1, 1, 0))])
def test_pcg_3d_chunk_depths(oracle_mod, n, periodic, precision):
    from cajitafluids_amd import _lib
    from cajitafluids_amd.solver import Solver
    cfg = K.base_config(3, n[0])
    cfg.update(num_cell=list(n), hi=[1.0, n[1] / n[0], n[2] / n[0]], clamp_dt=0, dt=0.002,
               halo=1, field_order=1, periodic=list(periodic), precision=precision,
               cg_max_iter=5, cg_tol=1e-30, refine_mode=K.REFINE_RESTART, inner_max_iter=0)
    print(f"pcg chunks: {n} {periodic} {precision}", flush=True)
    sol, orc = Solver(cfg), oracle_mod.Oracle(cfg)
    sol.init_random_faces(5)
    gpu_to_oracle(sol, orc)
    for o in (sol, orc):
        o.build_rhs()
        o.rhs_remove_mean()
    with pytest.raises(_lib.CfError) as ei:
        sol.pressure_solve(precision)
    assert ei.value.code == _lib.CF_ENOCONV
    rc, st_o = orc.pressure_solve(precision)
    assert rc == _lib.CF_ENOCONV
    assert sol.last_stats["iterations"] == st_o["iterations"]
    x_g = sol.owned_view(sol.get_pressure(0), 0)
    x_o = orc.owned_view(orc.lhs(), 0)
    assert np.any(x_o != 0.0)
    assert np.array_equal(x_g, x_o)
    sol.close()
    orc.close()
