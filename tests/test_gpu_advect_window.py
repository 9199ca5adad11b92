"""The 3-D advection kernel with its velocity window in LDS: one time
integration bit for bit the oracle's, at the edges of its 32 x 4 x 4 blocks
(full blocks, whose wall face layer is taken apart, and remainders of one and
of all but one), axes shorter than the window's reach, periodic and wall
axes, steps short and longer than the window, and non-finite velocities."""
import numpy as np
import pytest

from cajitafluids_amd import configs as K
from helpers import gpu_to_oracle

pytestmark = pytest.mark.gpu

# 256 blocks and more, but for the last grid (252, the general kernel)
GRIDS = [
    ((32, 64, 64), (0, 0, 0)), ((64, 32, 64), (0, 1, 0)), ((31, 63, 61), (0, 0, 0)),
    ((33, 33, 60), (1, 0, 0)), ((3, 3, 1024), (1, 1, 1)), ((2, 1, 1023), (0, 0, 0)),
    ((1030, 13, 7), (0, 0, 1)), ((65, 6, 170), (1, 1, 1)), ((32, 36, 112), (0, 0, 0)),
]


@pytest.mark.parametrize("order,halo", [(3, 3), (3, 2), (1, 1)])
@pytest.mark.parametrize("n,periodic", GRIDS)
@pytest.mark.parametrize("case", ["short", "long", "nonfinite"])
def test_advect_window(oracle_mod, n, periodic, order, halo, case):
    from cajitafluids_amd.solver import Solver
    if any(p and m < halo for p, m in zip(periodic, n)):
        pytest.skip("a periodic axis needs at least halo cells")
    cfg = K.base_config(3, n[0])
    # random faces are in [-1, 1]: steps of up to half a cell, or of six
    dt = (6.0 if case == "long" else 0.5) / n[0]
    cfg.update(num_cell=list(n), hi=[1.0, n[1] / n[0], n[2] / n[0]], clamp_dt=0, dt=dt,
               halo=halo, field_order=order, velocity_order=1, periodic=list(periodic))
    print(f"advect window: {n} {periodic} order {order} halo {halo} {case}", flush=True)
    sol, orc = Solver(cfg), oracle_mod.Oracle(cfg)
    sol.init_random_faces(9)
    rng = np.random.default_rng(4)
    q = sol.get(0)
    q[...] = rng.standard_normal(q.shape)
    sol.set(0, q)
    if case == "nonfinite":
        for e, bad in ((1, np.nan), (2, np.inf), (3, -np.inf)):
            f = sol.get(e)
            own = sol.owned_view(f, e)
            own[tuple(s // 2 for s in own.shape)] = bad
            sol.set(e, f)
    gpu_to_oracle(sol, orc)
    sol.time_integrate()
    orc.time_integrate()
    for e in range(4):
        g = sol.owned_view(sol.get(e), e)
        o = orc.owned_view(orc.field(e), e)
        assert np.array_equal(g, o, equal_nan=True), f"entity {e}"
    sol.close()
    orc.close()
