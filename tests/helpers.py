"""Seeded synthetic inputs shared by the tests (generated by the oracle's
splitmix64/Box-Muller stream, so GPU and CPU paths see identical bytes)."""
import ctypes
import functools
import os
import subprocess
import tempfile

import numpy as np

import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256  # MI355X
W144, RAW, Q6 = 0, 1, 2  # the prefill GEMMs' tiers


def weights(seed, N, K, qtype="q5k", std=0.02):
    w = O.gaussian(seed, N * K, 0.0, std).reshape(N, K)
    return O.quantize_q5k(w) if qtype == "q5k" else O.quantize_q6k(w)


def acts(seed, M, K):
    x = O.gaussian(seed, M * K, 0.0, 1.0).reshape(M, K)
    return x, O.q8_rows(x)


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    return t.detach().cpu().numpy()


# independent numpy decoders of the GGUF layouts (vectorised, written from the
# published block layouts: Q5_K d, dmin, scales[12], qh[32], qs[128]; Q6_K
# ql[128], qh[64], sc[16], d)
def np_codes_q5k(raw, K):
    """5-bit codes (0..31) of every value, [N][K]."""
    N = raw.shape[0]
    b = raw.reshape(N, K // 256, 176)
    qh = b[:, :, 16:48]
    qs = b[:, :, 48:176].reshape(N, K // 256, 4, 32)
    out = np.empty((N, K // 256, 8, 32), np.int32)
    for j in range(8):
        nib = (qs[:, :, j // 2, :] >> (4 * (j % 2))) & 0xF
        out[:, :, j, :] = nib | (((qh >> j) & 1) << 4)
    return out.reshape(N, K)


def np_codes_q6k(raw, K):
    """6-bit codes (0..63, before the -32 offset) of every value, [N][K]."""
    N = raw.shape[0]
    b = raw.reshape(N, K // 256, 210)
    ql = b[:, :, :128].reshape(N, K // 256, 2, 2, 32)   # [half][u&1][l]
    qh = b[:, :, 128:192].reshape(N, K // 256, 2, 32)
    out = np.empty((N, K // 256, 2, 4, 32), np.int32)
    for u in range(4):
        lo = (ql[:, :, :, u % 2, :] >> (4 * (u // 2))) & 0xF
        out[:, :, :, u, :] = lo | (((qh >> (2 * u)) & 3) << 4)
    return out.reshape(N, K)


def kat_q5k(N, K):
    """tools/mmq_test.cu:311-324 simple==3 blocks: d = 1, dmin = 0, scale
    bytes 01 01 01 01 | 00 00 00 00 | 11 11 11 11 (sc = 1 for all eight
    sub-blocks), qh = 0 and every code 1.  With x = 1, xd = 1, xsum = 0 every
    output is exactly K."""
    raw = np.zeros((N, K // 256, 176), np.uint8)
    raw[:, :, 0:2] = np.frombuffer(np.uint16(0x3C00).tobytes(), np.uint8)
    raw[:, :, 4:8] = 0x01
    raw[:, :, 12:16] = 0x11
    raw[:, :, 48:176] = 0x11
    return raw.reshape(N, -1)


def kat_q6k(N, K):
    """The same KAT for Q6_K: d = 1, every 16-value scale 1, every code 33
    (q - 32 = 1: low nibble 1 in both halves of each ql byte, high bits 2 in
    each 2-bit field of qh), so y = K for x = 1, xd = 1."""
    raw = np.zeros((N, K // 256, 210), np.uint8)
    raw[:, :, 0:128] = 0x11
    raw[:, :, 128:192] = 0xAA
    raw[:, :, 192:208] = 1
    raw[:, :, 208:210] = np.frombuffer(np.uint16(0x3C00).tobytes(), np.uint8)
    return raw.reshape(N, -1)


def check(oracle, y, ref, tol=1e-4, floor=1e-2, etol=1e-3, what=""):
    """The parity bar for fp32 outputs, both measures printed:
    * normwise per activation row, max |y - ref| / max |ref| of the row,
      below `tol` = 1e-4 (BASELINE's "max relative error 1e-4");
    * elementwise, |y - ref| / max(|ref|, floor x the row's max |ref|), below
      `etol` = 1e-3, the reference's own per-output bar (tools/mmq_test.cu:391:
      |y - ref| > 1e-3 |ref| + 1e-4 counts as bad).  Outputs far below the
      row's largest are cancellations of large terms whose fp32 rounding
      scales with the terms, hence the floor."""
    nw = oracle.normwise_err(y, ref)
    ew = oracle.elementwise_err(y, ref, floor)
    print(f"  parity {what}: normwise {nw:.2e}, elementwise (floor {floor:g}) {ew:.2e}", flush=True)
    assert nw < tol, (what, nw)
    assert ew < etol, (what, ew)
    return nw, ew


@functools.lru_cache(maxsize=None)
def mmq_plan():
    """The prefill GEMMs' launch choice and deal (bq_mmq_plan.hpp behind
    tests/host/mmq_plan.cpp), built with the host compiler."""
    tmp = tempfile.TemporaryDirectory()
    so = os.path.join(tmp.name, "mmq_plan.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "bruce-engine_amd", "csrc"), os.path.join(ROOT, "tests", "host", "mmq_plan.cpp"),
                    "-o", so], check=True)
    L = ctypes.CDLL(so)
    I, S, P = ctypes.c_int, ctypes.c_size_t, ctypes.POINTER(ctypes.c_int)
    L.t_pick.argtypes, L.t_pick.restype = [I, I, I, I, S, I, P], None
    L.t_ws_floats.argtypes, L.t_ws_floats.restype = [I, I, I, I], S
    L.t_reserved_differs.argtypes, L.t_reserved_differs.restype = [I, I, I, I, I, P], ctypes.c_long
    L.t_deal.argtypes, L.t_deal.restype = [I] * 6, I
    L.t_div.argtypes, L.t_div.restype = [I, I, P], None
    return L


def mmq_launch(tier, K, N, rows, ws_floats=None):
    """(token-tile height, K slices, slices per leftover tile, leftover tiles) of
    the launch a prefill GEMM takes on MI355X; ws_floats None: the reserved workspace."""
    L = mmq_plan()
    out = (ctypes.c_int * 4)()
    ws = L.t_ws_floats(rows, K, N, CUS) if ws_floats is None else ws_floats
    L.t_pick(tier, rows, K, N, ws, CUS, out)
    return tuple(out)
