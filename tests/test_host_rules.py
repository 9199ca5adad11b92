"""The rules by which the library chooses kernels on the host, called on the
CPU (tests/native/host_rules.cpp against the built library): the grids of the
GPU tests run the kernels that those tests are for."""
import os
import subprocess

import pytest

import test_gpu_mg_waves as waves

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("native") / "host_rules")
    lib = os.path.join(REPO, "cajitafluids_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(REPO, "include"), "-I" + os.path.join(lib, "csrc"),
                    "-o", exe, os.path.join(REPO, "tests", "native", "host_rules.cpp"),
                    "-L" + lib, "-lcfmi", "-L/opt/rocm/lib", "-lamdhip64",
                    "-Wl,-rpath," + lib + ":/opt/rocm/lib"], check=True)

    def call(*args):
        out = subprocess.run([exe, *map(str, args)], check=True, capture_output=True, text=True)
        return [int(v) for v in out.stdout.split()]

    return call


@pytest.mark.parametrize("n,periodic,precision,nu,want", waves.CASES)
def test_leg_waves(rules, n, periodic, precision, nu, want):
    level = list(n)
    for l, w in enumerate(want):
        boxes = l > 0 and any(m % 2 for m in n)
        f32 = precision == waves.K.FP32_REFINED and not boxes
        assert rules("leg", 3, *level, *periodic, nu, int(f32), int(boxes)) == [w], level
        level = [(m + 1) // 2 for m in level]


@pytest.mark.parametrize("dim,n,fits", [
    (2, (1, 1, 1), True), (2, (32, 32, 1), True), (2, (1024, 1024, 1), True),
    (2, (2337, 256, 1), True), (2, (2338, 10, 1), False), (2, (1200, 1200, 1), False),
    (3, (1, 1, 1), True), (3, (45, 52, 61), True), (3, (100, 100, 100), True),
    (3, (682, 20, 20), True), (3, (683, 2, 2), False), (3, (128, 128, 128), False),
    (3, (256, 256, 256), False)])
def test_coop_plan(rules, dim, n, fits):
    """A plan is made from the geometry alone, without a GPU, and handed to the
    launches; what fits: at most 256 workgroups of 4096 cells, whole x-rows."""
    groups, lds = rules("coop", dim, *n)
    cells = n[0] * n[1] * n[2]
    if fits:
        assert (cells + 4095) // 4096 <= groups <= 256
        assert 0 < lds <= 150 * 1024
    else:
        assert groups == 0


@pytest.mark.parametrize("dim,n,blocks,want", [
    (2, (128, 128, 1), 512, [1, 128, 1, 1, 128, 1]),  # 16 strips on every eighth block
    (2, (128, 128, 1), 96, [1, 16, 2, 1, 16, 1]),
    (2, (128, 128, 1), 15, [0, 16, 2, 0, 16, 1]),
    (2, (32, 32, 1), 1, [1, 1, 1, 1, 1, 1]),
    (3, (20, 20, 20), 1, [0, 16, 2, 0, 16, 1]),
    (3, (20, 20, 20), 16, [1, 16, 2, 1, 16, 1]),
])
def test_coop_spread(rules, dim, n, blocks, want):
    """A device that does not hold the idle blocks between the workgroups still
    runs the solve if it holds the workgroups."""
    assert rules("spread", dim, *n, blocks) == want
