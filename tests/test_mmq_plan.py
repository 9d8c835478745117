"""The prefill GEMMs' launch choice (bq_mmq_plan.hpp: token-tile height, K
split, leftover-tile split) on the CPU: it depends on the shape alone as long as
the caller holds the workspace bq_gemm_workspace_bytes reserves.  Under the
reserved size every launch must be the one an unlimited workspace gives, or
equal calls would take another path (another summation order) once a larger
workspace is at hand.  And the deal of a launch's blocks: every tile and K slice
once, in the order the kernels count on."""
import ctypes

import pytest

import test_gpu_raw_stages
import test_gpu_tile_order
from helpers import CUS, Q6, RAW, W144, mmq_launch, mmq_plan


@pytest.fixture(scope="module")
def picker():
    return mmq_plan()


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
    assert mmq_launch(tier, K, N, rows)[:3] == (tm, ks, tail)


def test_measured_case_launches():
    """The GPU tests of the tile order and of the raw tier's staging name the
    launch each case is there for: the choice still takes it, and together they
    run both heights of every tier whole and K-split and both of the Q5_K
    tiers' leftover splits, each in the grouped order with a narrow last group."""
    seen = set()
    for fmt, K, Ns, rows, launch in test_gpu_tile_order.CASES:
        tier = {"q5k_rep": W144, "q5k": RAW, "q6k_rep": Q6}[fmt]
        tm, ks, tail, left = mmq_launch(tier, K, sum(Ns), rows)
        assert (tm, ks, tail) == launch, (fmt, K, Ns, rows)
        ntm, ntn, group, rnd = -(-rows // tm), sum(Ns) // 128, *((4, 24) if tm == 32 else (8, 8))
        if ntm > rnd and ntn % group:
            seen.add((tier, tm, "tail" if tail > 1 else "split" if ks > 1 else "whole"))
            if tail > 1:  # leftover tiles inside the narrow group
                assert left <= ntm * (ntn % group)
    for K, N, rows, launch in test_gpu_raw_stages.CASES:
        assert mmq_launch(RAW, K, N, rows)[:3] == launch, (K, N, rows)
    want = {(t, tm, m) for t in (W144, RAW, Q6) for tm in (32, 128) for m in ("whole", "split", "tail")}
    assert seen == want - {(Q6, 32, "tail"), (Q6, 128, "tail")}


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
