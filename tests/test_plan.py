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
extern "C" void plan(int64_t m, int64_t n, int64_t k, int S, int K, int rg, int64_t cap, int cus, int* out) {
    const LinPlan p = linear_plan(m, n, k, S, K, rg, cap, cus);
    out[0] = p.RG;
    out[1] = p.P;
    out[2] = p.bps;
}
extern "C" int64_t call_bytes(int64_t m, int64_t n, int64_t k, int S, int K, int cus, uint64_t most) {
    LinPlan p;
    return linear_call_plan(m, n, k, S, K, 0, cus, most, &p) ? (int64_t)linear_call_bytes(m, n, k, S, p.P) : -1;
}
extern "C" int few_rows(int64_t m, int64_t n, int64_t k, int K) { return linear_few_rows(m, n, k, K); }
extern "C" int router(int64_t M, int64_t E) { return router_rows(M, E, 256); }
extern "C" int64_t max_blocks(int64_t npairs, int64_t E, int rows, int whole) { return moe_max_blocks(npairs, E, rows, whole); }
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
    L.plan.argtypes = [i64, i64, i64, i32, i32, i32, i64, i32, ctypes.c_void_p]
    L.plan.restype = None
    L.moe_rows.argtypes = [i64] * 5 + [i32] * 3
    L.moe_rows.restype = i32
    L.call_bytes.argtypes = [i64, i64, i64, i32, i32, i32, ctypes.c_uint64]
    L.call_bytes.restype = i64
    L.few_rows.argtypes = [i64, i64, i64, i32]
    L.few_rows.restype = i32
    L.router.argtypes = [i64, i64]
    L.router.restype = i32
    L.max_blocks.argtypes = [i64, i64, i32, i32]
    L.max_blocks.restype = i64
    return L


def plan(lib, m, n, k, K, rg=0, cap=1 << 30, S=1):
    out = (ctypes.c_int * 3)()
    lib.plan(m, n, k, S, K, rg, cap, CUS, out)
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


SHAPES = [(1024, 4096), (4096, 4096), (4096, 14336), (5376, 21504), (21504, 5376), (2048, 131072), (8192, 1024), (12288, 128)]


def gemv_bytes(m, n, k):
    """The decode GEMV's partials (csrc/exl3_linear.hip: gemv_splits, gemv_part_bytes)."""
    strips, nblk = n // 128, k // 128
    P = min(-(-1024 // strips), 8 if m <= 2 else 16)
    return strips * max(1, min(max(P, -(-nblk // 8)), nblk)) * 8 * 128 * 4


@pytest.mark.parametrize("k,n", SHAPES)
@pytest.mark.parametrize("S", [1, 3, 64])
def test_few_rows_keep_to_the_gemv_scratch(lib, k, n, S):
    """Five to eight rows on the MFMA GEMM never need more scratch than the GEMV that they replace, so that the choice can
    follow from the shape alone; with one shard they always fit."""
    for m in range(5, 9):
        for K in range(1, 9):
            b = lib.call_bytes(m, n, k, S, K, CUS, gemv_bytes(m, n, k))
            assert b <= gemv_bytes(m, n, k)
            assert b > 0 or S > 1 or n < 4096


@pytest.mark.parametrize("k,n", SHAPES)
def test_call_scratch_is_bounded(lib, k, n):
    """Partials of at most as many splits as fill the device with blocks of 16, 32 or 64 rows (4, 3 or 2 workgroups per CU)."""
    for m in (9, 16, 17, 32, 33, 100, 512, 2048):
        rows, per_cu = (16, 4) if m <= 16 else (32, 3) if m <= 32 else (64, 2)
        nblk, tiles = k // 128, -(-m // rows) * -(-n // 256)
        P = min(-(-per_cu * CUS // tiles), max(1, nblk // 2))
        P = -(-nblk // -(-nblk // P))
        up = lambda v: -(-v // 256) * 256  # noqa: E731
        for S in (1, 3):
            most = up(2 * S * m * k) + up(4 * S * m * nblk) + (up(4 * P * m * n) if P > 1 else 0)
            for K in (2, 4, 6, 8):
                assert lib.call_bytes(m, n, k, S, K, CUS, 1 << 62) <= most


def blocks_of(c, rows, whole):
    """Row blocks of an expert with c rows (BlockCut in csrc/exl3_moe.h)."""
    full, rem = divmod(c, rows)
    return full + (-(-rem // 32) if rows > 64 and not whole and rem <= 64 else rem > 0)


@pytest.mark.parametrize("rows,whole", [(32, False), (64, False), (128, False), (64, True), (128, True)])
def test_block_list_holds_every_routing(lib, rows, whole):
    for c in range(1, 600):
        for E in (1, 2, 7):
            assert E * blocks_of(c, rows, whole) <= lib.max_blocks(E * c, E, rows, whole)
    assert blocks_of(33, rows, whole) + 5 * blocks_of(1, rows, whole) <= lib.max_blocks(38, 6, rows, whole)


def test_few_rows_take_the_gemm_where_it_is_faster(lib):
    """Both sides of the measured lines: by size, by rows and by bitrate."""
    for m, K, k, n, want in ((4, 4, 5376, 21504, 0), (5, 4, 8192, 8192, 1), (5, 4, 4096, 14336, 0), (8, 4, 4096, 8192, 0),
                             (8, 4, 4096, 11008, 1), (6, 5, 4096, 12288, 1), (6, 6, 4096, 12288, 0), (6, 6, 4096, 14336, 1),
                             (6, 7, 8192, 8192, 0), (7, 7, 8192, 8192, 1), (7, 8, 8192, 8192, 0), (8, 8, 4096, 14336, 1),
                             (5, 8, 5376, 21504, 1), (9, 4, 5376, 21504, 0)):
        assert lib.few_rows(m, n, k, K) == want, (m, K, k, n)


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("rg", [0, 4])
def test_no_spilling_row_block(lib, K, rg):
    """128-row blocks of several shards spill registers inside their loop for K > 5: not picked, not even when asked for."""
    for k, n in ((1024, 3072), (4096, 6144), (5376, 10752), (8192, 2048)):
        for m in (77, 128, 300, 397, 512, 800, 1024, 1500, 2048):
            RG = plan(lib, m, n, k, K, rg, 2 * CUS, 3)[0]
            assert RG != 4 or K <= 5
            assert rg == 0 or RG == (4 if K <= 5 else 2)


@pytest.mark.parametrize("M,H,I", [(40, 8192, 2048), (300, 1024, 2048)])
def test_dense_mlp_capture_shapes_have_many_splits(lib, M, H, I):
    """The shapes of test_dense_mlp_captured_in_the_scratch_of_an_unsplit_call have several splits, more than the one set of
    partials that its workspace holds."""
    rows = lib.moe_rows(M, 1, M, H, I, 3, 3, 0)
    assert plan(lib, M, H, I, 3, rows // 32, 8)[1] > 2


def test_router_rows_by_rounds(lib):
    """Rows per workgroup of the router GEMV: few while every CU has at most one workgroup, more before a second round."""
    for M, E, want in ((1, 512, 1), (8, 512, 1), (32, 512, 1), (48, 512, 2), (64, 512, 2), (96, 512, 4), (200, 160, 4),
                       (256, 160, 4), (128, 256, 2), (200, 256, 4), (512, 8, 2), (512, 160, 2), (4 * 65535, 8, 4)):
        assert lib.router(M, E) == want, (M, E)
        assert -(-M // lib.router(M, E)) <= 65535              # the grid's second dimension


def test_row_block_by_load(lib):
    """Row blocks of the prefill MoE by batch and load, at the sizes of the blob tests among others."""
    for M, E, slots, K, want in ((160, 6, 2, 3, 64), (480, 12, 2, 3, 128), (700, 6, 2, 5, 128), (700, 6, 2, 6, 64),
                                 (64, 16, 8, 3, 32), (160, 256, 8, 3, 32), (160, 64, 8, 3, 128), (512, 160, 8, 2, 128),
                                 (1024, 512, 10, 3, 128), (40, 1, 1, 4, 64), (397, 1, 1, 4, 128), (397, 1, 1, 8, 64)):
        assert lib.moe_rows(M, E, M * slots, 2048, 1024, K, K, 0) == want, (M, E, slots, K)
