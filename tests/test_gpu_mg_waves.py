"""The 3-D multigrid legs in blocks of 16 and of 12 waves with two and three
sweeps, against the oracle's V-cycle: FP64 levels of one coupling (16) and of
boxes (12); FP32 finest levels (16) above an FP64 level of boxes, and above an
FP32 level that runs in 16 waves too.  test_host_rules.py holds the blocks'
waves on the first two levels, which CASES lists."""
import pytest

from cajitafluids_amd import configs as K
from test_gpu_mg_legs import check_solve

pytestmark = pytest.mark.gpu

# cells, periodic axes, precision, sweeps, waves of the first two levels' blocks
CASES = [
    ((129, 121, 97), (0, 0, 0), K.FP32_REFINED, 2, (16, 8)),
    ((129, 121, 97), (0, 0, 0), K.FP32_REFINED, 3, (16, 8)),
    ((190, 182, 149), (1, 1, 0), K.FP32_REFINED, 2, (16, 8)),
    ((190, 182, 149), (1, 1, 0), K.FP32_REFINED, 3, (16, 8)),
    ((252, 244, 164), (0, 0, 0), K.FP32_REFINED, 2, (16, 16)),
    ((252, 244, 164), (0, 0, 0), K.FP32_REFINED, 3, (16, 16)),
    ((130, 121, 96), (0, 1, 0), K.FP64, 2, (16, 8)),
    ((247, 83, 499), (0, 0, 0), K.FP64, 2, (16, 12)),
    ((247, 243, 159), (1, 0, 0), K.FP64, 3, (16, 12)),
]


@pytest.mark.parametrize("n,periodic,precision,nu,waves", CASES)
def test_mg_leg_waves(oracle_mod, n, periodic, precision, nu, waves):
    check_solve(oracle_mod, n, periodic, nu, precision)
