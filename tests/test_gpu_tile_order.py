"""The prefill GEMMs' grouped tile order (bq_gemm.hip tile_at) at the sizes
where it can go wrong: more token tiles than one round (24 of 32 tokens, 8 of
128; below that the order is panel-major), a last panel group narrower than the
others, a ragged last token tile, several parts, launches whose leftover tiles
run as K slices, and launches split over K whose pieces the XCDs share unevenly
(map_tile: ranges that start and end inside a tile).  Every output
is compared with the oracle of its tier (helpers.check), so a tile that is
skipped, written twice from another tile's operands, or summed into another
tile's place shows."""
import numpy as np
import pytest

from helpers import acts, check, dev, host, weights

pytestmark = pytest.mark.gpu

CASES = [
    # fmt, K, Ns, rows
    ("q5k_rep", 512, [1408, 640], 1157),   # 16 panels; 32-token tiles: 37 token tiles, leftover split
    ("q5k_rep", 512, [1152], 1290),        # 9 panels: a last group of one
    ("q5k", 256, [896, 256], 1157),        # raw tier
    ("q6k_rep", 512, [1664], 1157),        # 13 panels: a last group of five
    ("q5k_rep", 512, [384], 801),          # 26 token tiles of 32, fewer panels than a group
    ("q6k_rep", 1792, [1664], 70),         # K slices over 13 x 3 tiles
    ("q5k_rep", 2560, [1408], 300),        # K slices over 11 x 10 tiles
    ("q5k", 1280, [896, 256], 150),        # raw tier, K slices over 9 x 5 tiles
]


@pytest.mark.parametrize("fmt,K,Ns,rows", CASES)
def test_every_tile_in_its_place(bq, oracle, fmt, K, Ns, rows):
    import torch
    print(f"tile order {fmt} K={K} Ns={Ns} rows={rows}", flush=True)
    q5 = fmt.startswith("q5k")
    raws = [weights(700 + p + K + n, n, K, "q5k" if q5 else "q6k") for p, n in enumerate(Ns)]
    _, (xq, xd, xs) = acts(711 + rows, rows, K)
    ws, refs = [], []
    for raw, n in zip(raws, Ns):
        g = dev(raw)
        if fmt == "q5k_rep":
            w144, dm = bq.repack_q5k(g, K, n)
            ws.append(bq.make_weight(g, bq.TYPE_Q5_K, K, n, rep=w144, rep_min=dm))
            r144, rdm = oracle.repack_q5k_144(raw, K)
            refs.append(oracle.gemm_q5k_144(r144, rdm, xq, xd, oracle.fill_xdh(xd, xs), n))
        elif q5:
            ws.append(bq.make_weight(g, bq.TYPE_Q5_K, K, n))
            refs.append(oracle.gemm_q5k(raw, xq, xd, xs))
        else:
            ws.append(bq.make_weight(g, bq.TYPE_Q6_K, K, n, rep=bq.repack_q6k(g, K, n)))
            refs.append(oracle.gemm_q6k(raw, xq, xd))
    ys = [torch.full((rows, n), float("nan"), device="cuda") for n in Ns]
    xdh = torch.zeros((rows, K // 32), dtype=torch.int16, device="cuda")
    bq.gemm_b_fused(ys, ws, rows, dev(xq), dev(xd), dev(xs), xdh)
    torch.cuda.synchronize()
    for p, (y, ref) in enumerate(zip(ys, refs)):
        check(oracle, host(y), ref, what=f"{fmt} part {p}")
