"""The wide-block kernels' host-side choices (csrc/exl3_plan.h, plain C++), compiled here and checked without a GPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "b70-inference_amd", "csrc")
CUS = 256

SHIM = """
#include "exl3_plan.h"
using namespace exl3;
extern "C" void plan(int64_t m, int64_t n, int64_t k, int K, int rg, int64_t cap, int cus, int* out) {
    const LinPlan p = linear_plan(m, n, k, K, rg, cap, cus);
    out[0] = p.RG;
    out[1] = p.P;
    out[2] = p.bps;
}
extern "C" int moe_rows(int64_t M, int64_t E, int64_t npairs, int64_t H, int64_t I, int Kg, int Kd, int forced) {
    return moe_wide_rows(M, E, npairs, H, I, Kg, Kd, forced);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.check_call([cxx, "-std=c++20", "-O1", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(d / "plan.so"),
                           str(d / "shim.cpp")])
    L = ctypes.CDLL(str(d / "plan.so"))
    i64, i32 = ctypes.c_int64, ctypes.c_int
    L.plan.argtypes = [i64, i64, i64, i32, i32, i64, i32, ctypes.c_void_p]
    L.plan.restype = None
    L.moe_rows.argtypes = [i64] * 5 + [i32] * 3
    L.moe_rows.restype = i32
    return L


def plan(lib, m, n, k, K, rg=0, cap=1 << 30):
    out = (ctypes.c_int * 3)()
    lib.plan(m, n, k, K, rg, cap, CUS, out)
    return list(out)


def last_byte(rows, k):
    """Past the last byte that a workgroup loads of a block's A, `rows` rows over k columns: steps of 32 columns take
    64 * rows bytes, and the loads of the last one end at its end."""
    return (k // 32) * 64 * rows


@pytest.mark.parametrize("k", [128, 4096, 1 << 22, (1 << 22) + 128, 65535 * 128])
@pytest.mark.parametrize("m", [9, 33, 100, 255, 256, 2048])
@pytest.mark.parametrize("rg", [0, 1, 2, 4, 8])
def test_linear_block_offsets_fit_32_bits(lib, m, k, rg):
    """Every A load of a block stays inside the 2^31 - 1 bytes that a buffer load reaches (zeros past them), also at the
    largest k that a call accepts and with a forced row block."""
    for n in (128, 16384):
        for cap in (1, 4):
            RG, P, bps = plan(lib, m, n, k, 1, rg, cap)
            assert P == -(-(k // 128) // bps) and 1 <= P <= cap
            assert RG in (1, 2, 4, 8) and (rg == 0 or RG <= rg)
            assert last_byte(min(m, 32 * RG), min(k, 128 * bps)) <= (1 << 31) - 1


@pytest.mark.parametrize("width", [128, 1 << 22, (1 << 23) - 128, 1 << 23, 1 << 24])
@pytest.mark.parametrize("forced", [0, 64, 128])
def test_moe_block_offsets_fit_32_bits(lib, width, forced):
    for H, I in ((128, width), (width, 128)):
        for M, E, slots in ((200, 1, 1), (2048, 1, 1), (2048, 8, 2), (300, 64, 8)):
            rows = lib.moe_rows(M, E, M * slots, H, I, 2, 2, forced)
            assert rows in (32, 64, 128)
            assert last_byte(rows, width) <= (1 << 31) - 1
