"""Launch counts of HSMAC in divergence form (lcs_hsmac_plan.h), on the host.

Every pass that leaves a partial sum per workgroup has to fit a partial slot,
and every shell kernel its 32-bit index, for each box the form takes: cubes
and flat boxes beyond the sizes any test runs, and one cell either side of the
limits.  Boxes the form cannot do are left to the in-place sweeps."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build_native(tmp_path_factory, name):
    if not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("HIP headers not installed")
    out = tmp_path_factory.mktemp(name) / f"lib{name}.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "lcs.jl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", name + ".cpp"), "-o", str(out)], check=True)
    return C.CDLL(str(out))


@pytest.fixture(scope="module")
def plan_lib(tmp_path_factory):
    return build_native(tmp_path_factory, "hsmac_div_plan")


def plan(lib, dims, h, esize):
    out = (C.c_long * 13)()
    return list(out) if lib.hsmac_div_plan(*dims, h, esize, out) else None


TAKEN = [(8, 8, 8), (32, 32, 32), (1000, 1000, 1000), (1443, 1443, 1443), (1444, 1444, 1444), (1500, 1500, 1500),
         (2048, 2048, 64), (2048, 1024, 64), (2041, 2041, 8), (2042, 2043, 8), (4000, 4000, 8), (100, 4000, 4000),
         (4000, 8, 4000), (16000, 8, 8), (8, 16000, 8), (8, 8, 16000)]


@pytest.mark.parametrize("esize", [4, 8])
@pytest.mark.parametrize("dims", TAKEN)
@pytest.mark.parametrize("h", [3, 5])
def test_counts_fit(plan_lib, dims, h, esize):
    p = plan(plan_lib, dims, h, esize)
    assert p is not None
    cap, passes = p[0], p[1:5] + p[6:9]
    assert all(1 <= n <= cap for n in passes), p
    assert p[5] * 256 >= (dims[0] + 2 * h) * (dims[1] + 2 * h) and p[5] < 2**31
    assert max(p[9:12]) + cap * 256 < 2**31


def test_boxes_left_to_the_in_place_sweeps(plan_lib):
    for esize in (4, 8):
        for dims, h in [((7, 8, 8), 3), ((8, 8, 8), 2), ((8, 16, 16), 9),
                        ((20000, 20000, 8), 3),     # columns of tiles beyond a partial slot
                        ((16384, 8, 16400), 3)]:    # shell cells beyond 32-bit indices
            assert plan(plan_lib, dims, h, esize) is None, (dims, h, esize)
