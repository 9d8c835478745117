"""The prefill GEMMs' launch choice (bq_mmq_plan.hpp: token-tile height, K
split, leftover-tile split) on the CPU: it depends on the shape alone as long as
the caller holds the workspace bq_gemm_workspace_bytes reserves.  Under the
reserved size every launch must be the one an unlimited workspace gives, or
equal calls would take another path (another summation order) once a larger
workspace is at hand."""
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
