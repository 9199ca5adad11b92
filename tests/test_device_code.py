"""The machine code of the built library (csrc/check_code.py): the check finds
what it is for in listings written here, and nothing in the library."""
import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "cajitafluids_amd", "csrc")
if CSRC not in sys.path:
    sys.path.insert(0, CSRC)

import check_code  # noqa: E402


@pytest.fixture(scope="module")
def listings():
    path = os.environ.get("CFMI_LIBRARY", os.path.join(REPO, "cajitafluids_amd", "libcfmi.so"))
    out = [check_code.disassemble(c) for c in check_code.code_objects(path)]
    kernels = {t for lines in out for t in lines if t.startswith("<_ZN4cfmi")}
    assert any("k_advect_win" in k for k in kernels)
    assert any("k_pcg_solve_coop3" in k for k in kernels)
    return out


@pytest.mark.parametrize("between,found", [
    ([], 1), (["s_barrier"], 0), (["s_nop 0"], 0), (["v_mov_b32_e32 v9, v8"], 0),
])
def test_lane_read_after_its_write(between, found):
    code = ["<_Z1kv>:", "v_mul_f64 v[36:37], v[36:37], 0.5", *between,
            "v_readfirstlane_b32 s50, v37"]
    assert len(check_code.lane_read_hazards(code)) == found


@pytest.mark.parametrize("between,found", [
    ([], 1), (["s_nop 0"], 1), (["s_nop 1"], 0), (["s_add_i32 s1, s1, 1", "s_barrier"], 0),
])
def test_use_after_lane_read(between, found):
    code = ["<_Z1kv>:", "v_readlane_b32 s50, v1, 3", *between,
            "v_add_f64 v[2:3], v[2:3], s[50:51]"]
    assert len(check_code.lane_read_hazards(code)) == found


def test_library_lane_reads(listings):
    assert [h for lines in listings for h in check_code.lane_read_hazards(lines)] == []
