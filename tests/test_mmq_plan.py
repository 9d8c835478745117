"""The prefill GEMMs' launch choice (bq_mmq_plan.hpp: token-tile height, K
split, leftover-tile split) on the CPU: it depends on the shape alone as long as
the caller holds the workspace bq_gemm_workspace_bytes reserves.  Under the
reserved size every launch must be the one an unlimited workspace gives, or
equal calls would take another path (another summation order) once a larger
workspace is at hand.  And the deal of a launch's blocks: every tile and K slice
once, in the order the kernels count on."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
W144, RAW, Q6 = 0, 1, 2
CUS = 256  # MI355X


@pytest.fixture(scope="module")
def picker(tmp_path_factory):
    so = tmp_path_factory.mktemp("mmq_plan") / "mmq_plan.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "bruce-engine_amd", "csrc"), os.path.join(ROOT, "tests", "host", "mmq_plan.cpp"),
                    "-o", str(so)], check=True)
    L = ctypes.CDLL(str(so))
    I, S, P = ctypes.c_int, ctypes.c_size_t, ctypes.POINTER(ctypes.c_int)
    L.t_pick.argtypes, L.t_pick.restype = [I, I, I, I, S, I, P], None
    L.t_ws_floats.argtypes, L.t_ws_floats.restype = [I, I, I, I], S
    L.t_reserved_differs.argtypes, L.t_reserved_differs.restype = [I, I, I, I, I, P], ctypes.c_long
    L.t_deal.argtypes, L.t_deal.restype = [I] * 6, I
    L.t_div.argtypes, L.t_div.restype = [I, I, P], None
    return L


@pytest.mark.parametrize("tier,k_step", [(W144, 512), (RAW, 256), (Q6, 256)])
@pytest.mark.parametrize("cus", [CUS, 304])
def test_reserved_workspace_gives_the_unlimited_launch(picker, tier, k_step, cus):
    first = (ctypes.c_int * 4)()
    bad = picker.t_reserved_differs(tier, cus, k_step, 384, 8192, first)
    assert bad == 0, (bad, list(first))


def test_reserved_workspace_of_short_raw_k(picker):
    """Raw Q5_K at K = 768: the 32-token tile's leftover split saves just more
    than it must, so the reserve has to weigh it as the launch does."""
    out = (ctypes.c_int * 4)()
    for N, rows in ((2048, 2120), (1408, 3000), (2176, 2048)):
        ws = picker.t_ws_floats(rows, 768, N, CUS)
        picker.t_pick(RAW, rows, 768, N, ws, CUS, out)
        under = list(out)
        picker.t_pick(RAW, rows, 768, N, ctypes.c_size_t(-1).value, CUS, out)
        assert under == list(out), (N, rows)


# Launches measured at every height and split: the fastest one (token-tile height,
# K slices, slices per leftover tile), its time, and the time of the launch an
# estimate fitted to nine shapes took instead (us).
MEASURED = [
    # tier, K, N, rows, height, slices, leftover slices
    (W144, 3072, 9216, 905, 128, 1, 4),     # 85.0, was 91.0
    (W144, 3072, 9216, 1279, 128, 1, 1),    # 110.8, was 119.6
    (W144, 4096, 3072, 3717, 128, 1, 1),    # 144.1, was 156.0
    (W144, 6144, 16640, 1128, 128, 1, 1),   # 325.5, was 369.2
    (W144, 7168, 2560, 3268, 128, 1, 4),    # 172.8, was 193.3
    (W144, 2560, 14336, 1281, 128, 1, 1),   # 147.1, was 161.4
    (RAW, 2048, 6912, 247, 32, 1, 1),       # 26.5, was 31.8
    (Q6, 8960, 3200, 253, 32, 3, 1),        # 49.3, was 57.0
    (Q6, 768, 9216, 3040, 128, 1, 1),       # 108.6, was 120.6
    (Q6, 8448, 8320, 3266, 128, 1, 1),      # 999, was 1095
]


@pytest.mark.parametrize("tier,K,N,rows,tm,ks,tail", MEASURED)
def test_measured_fastest_launch(picker, tier, K, N, rows, tm, ks, tail):
    out = (ctypes.c_int * 4)()
    picker.t_pick(tier, rows, K, N, picker.t_ws_floats(rows, K, N, CUS), CUS, out)
    assert list(out)[:3] == [tm, ks, tail]


@pytest.mark.parametrize("tm", [32, 128])
def test_every_piece_once(picker, tm):
    """Whole and K-split launches on both sides of the grouped order's limit
    (24 / 8 token tiles), panel counts around the groups of 4 / 8."""
    for ntm in (1, 2, 3, 5, 7, 8, 9, 13, 23, 24, 25, 31, 64):
        for ntn in (1, 2, 3, 4, 5, 7, 8, 9, 11, 15, 16, 17, 56, 72, 73):
            for ks in range(1, 9):
                if ks == 1 or ntm * ntn * ks <= 3 * 304:
                    assert picker.t_deal(tm, ntm, ntn, ks, 1, 0) == 0, (ntm, ntn, ks)


@pytest.mark.parametrize("tm", [32, 128])
def test_leftover_split_pieces(picker, tm):
    for ntm, ntn in ((32, 25), (9, 72), (16, 72), (41, 13), (8, 67), (25, 21)):
        left = ntm * ntn % CUS
        for k in (2, 3, 4):
            assert picker.t_deal(tm, ntm, ntn, 1, k, left) == 0, (ntm, ntn, k)


def test_short_division(picker):
    """tile_div<true> over what a split launch asks of it: up to 3 pieces per CU."""
    first = (ctypes.c_int * 2)()
    picker.t_div(4096, 1025, first)
    assert first[0] == -1, list(first)
