"""HSMAC in divergence form on the host: its launch counts (lcs_hsmac_plan.h), and
its passes (lcs_hsmac_div.h, lcs_hsmac_shell.h) run thread by thread in the
kernels' barrier order, against the oracle.

Every pass that leaves a partial sum per workgroup has to fit a partial slot,
and every shell kernel its 32-bit index, for each box the form takes: cubes
and flat boxes beyond the sizes any test runs, and one cell either side of the
limits.  Boxes the form cannot do are left to the in-place sweeps."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import rand_halo
from oracle import oracle as O

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


# ---- the passes themselves -------------------------------------------------------
TOL = {np.float64: 1e-12, np.float32: 2e-5}  # the parity tests' bound of one call, of the largest value


@pytest.fixture(scope="module")
def emul(tmp_path_factory):
    return build_native(tmp_path_factory, "hsmac_div_emul")


def run_emul(lib, A, h, dt, epsp, itrmin, itrmax, lf=None, shape=0, zc=7, stride=0):
    dims = [n - 2 * h for n in A[0].shape]
    itr, div, power = C.c_int(), C.c_double(), C.c_double()
    rc = lib.hsmac_div_emul(A[0].dtype.itemsize, *dims, h, (C.c_void_p * 4)(*[a.ctypes.data for a in A]),
                            C.c_double(dt), C.c_double(1.7), C.c_double(epsp), itrmin, itrmax,
                            None if lf is None else (C.c_double * 5)(*lf), shape, zc, stride, C.byref(itr),
                            C.byref(div), C.byref(power))
    assert rc == 0  # -1: not a box of this form, -2: written past an array
    return itr.value, div.value, power.value


# one window and several in x and y, the last one ending on and next to the array's
# end (58 + 6: a row of 64; 122 + 6: of 128), odd extents, padded rows (250 + 6), chunks
# of one plane to the whole depth, the smallest box, wider halos
CASES = [((8, 8, 8), 3, 0, 14), ((57, 9, 10), 3, 0, 3), ((58, 26, 9), 3, 0, 1), ((13, 64, 11), 3, 1, 6),
         ((121, 30, 8), 3, 2, 5), ((122, 50, 8), 3, 2, 14), ((250, 9, 8), 3, 1, 7), ((9, 12, 11), 4, 0, 4),
         ((40, 21, 12), 5, 1, 22), ((10, 9, 9), 9, 2, 9)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,h,shape,zc", CASES)
@pytest.mark.parametrize("itr", [1, 6])
def test_passes_on_the_host(emul, dims, h, shape, zc, itr, dtype):
    """Sweeps, refresh, face slabs and update against the oracle's in-place colour
    passes, ghosts included; the passes that stride give the same bits."""
    rng = np.random.default_rng(sum(dims) + h)
    A = [rand_halo(rng, dims, h, dtype) for _ in range(4)]
    B, S = ([a.copy(order="F") for a in A] for _ in range(2))
    got = run_emul(emul, B, h, 0.02, 1e-3, itr, itr, shape=shape, zc=zc)
    strided = run_emul(emul, S, h, 0.02, 1e-3, itr, itr, shape=shape, zc=zc, stride=1)
    n, div = O.hsmac(*A, h, 0.02, True, True, 0, 1.7, 1e-3, itr, itr)
    assert got[0] == strided[0] == n
    assert got[1] == pytest.approx(div, rel=1e-9 if dtype == np.float64 else 1e-4)
    for a, b, s in zip(A, B, S):
        assert np.abs(b - a).max() <= TOL[dtype] * np.abs(a).max()
        np.testing.assert_array_equal(b, s)


@pytest.mark.parametrize("itrmin,itrmax,epsp", [(30, 30, 0.0), (51, 60, 0.0), (0, 60, 1e-3), (6, 60, 1e-5)])
def test_forced_call_past_the_carry_on_the_host(emul, itrmin, itrmax, epsp):
    """Deferred linear forcing and the carry at 24 and 48 sweeps, calls that end
    by count and by epsp: U + A (U - mean) dt first, then the oracle's sweeps."""
    dims, h, dt, rng = (14, 11, 9), 3, 0.02, np.random.default_rng(3)
    lf = [0.0, 0.45, 0.55, 0.5, 1.3]
    A = [rand_halo(rng, dims, h) for _ in range(4)]
    B = [a.copy(order="F") for a in A]
    n, div, p = run_emul(emul, B, h, dt, epsp, itrmin, itrmax, lf=lf)
    power = 0.0
    for q in range(3):  # (the call fills the ghosts first, so theirs are forced alike)
        src = lf[4] * (A[q] - lf[1 + q])
        power += (A[q] * src)[h:-h, h:-h, h:-h].sum()
        A[q] += src * dt
    on, odiv = O.hsmac(*A, h, dt, True, True, 0, 1.7, epsp, itrmin, itrmax)
    assert n == on and (epsp == 0) == (n >= itrmax)
    assert div == pytest.approx(odiv, rel=1e-9)
    assert p == pytest.approx(power / np.prod(dims), rel=1e-12)
    for a, b in zip(A, B):
        assert np.abs(b - a).max() <= TOL[np.float64] * np.abs(a).max()
