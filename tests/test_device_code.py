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


JOIN = "s_or_b64 exec, exec, s[6:7]"


@pytest.mark.parametrize("opening,found", [
    (["v_mov_b32_e32 v26, v126"], 1), (["s_nop 0", "v_mov_b64_e32 v[2:3], v[8:9]"], 1),
    (["scratch_load_dword v26, off, off offset:16", "s_waitcnt vmcnt(0)"], 1), ([], 0),
    (["v_readlane_b32 s6, v40, 2", "v_readlane_b32 s7, v40, 3"], 0),
    (["v_mov_b32_e32 v26, v126", "v_add_u32_e32 v1, v26, v2"], 0),  # the block's own work
    (["v_mov_b32_e32 v26, v126", "s_cbranch_vccnz L2"], 0),
])
def test_move_before_a_join(opening, found):
    code = ["<_Z1kv>:", "s_and_saveexec_b64 s[6:7], vcc", "s_cbranch_execz L1",
            "v_mov_b32_e32 v5, v6", "<L1>:", *opening, JOIN, "v_mov_b32_e32 v7, v8"]
    assert len(check_code.early_moves(code)) == found


def test_library_joins(listings):
    joins = sum(a.startswith("<L") and b.startswith("s_or_b64 exec, exec,")
                for lines in listings for a, b in zip(lines, lines[1:]))
    assert joins > 100  # the listings show them as the check expects
    assert [m for lines in listings for m in check_code.early_moves(lines)] == []
