"""The prefill GEMMs' grouped tile order (bq_mmq_plan.hpp tile_at) at the sizes
where it can go wrong: more token tiles than one round (24 of 32 tokens, 8 of
128; below that the order is panel-major), a last panel group narrower than the
others (4 panels at 32 tokens, 8 at 128), a ragged last token tile, several
parts, launches whose leftover tiles run as K slices, and launches split over K
whose pieces the XCDs share unevenly (map_tile: ranges that start and end inside
a tile).  Every tile is compared with the oracle of its tier (helpers.check; of
the 128-token launches the first, a middle and the last row of every 32, all
columns), so a tile that is skipped, written twice from another tile's operands,
or summed into another tile's place shows.  Each case names the launch it is
there for (token-tile height, K slices, slices per leftover tile), which
test_mmq_plan.py checks without a GPU: a change of the launch choice cannot
take a case off its path unseen."""
import numpy as np
import pytest

from helpers import acts, check, dev, host, weights

pytestmark = pytest.mark.gpu

CASES = [
    # fmt, K, Ns, rows, launch
    ("q5k_rep", 512, [1408, 640], 1157, (32, 1, 1)),    # 16 panels x 37 token tiles, two parts
    ("q5k_rep", 512, [1152], 1290, (32, 1, 1)),         # 9 panels: a last group of one
    ("q5k", 256, [896, 256], 1157, (32, 1, 1)),         # raw tier, a last group of one
    ("q6k_rep", 512, [1664], 1157, (32, 1, 1)),         # 13 panels: a last group of one
    ("q5k_rep", 512, [384], 801, (32, 1, 1)),           # 26 token tiles, fewer panels than a group
    ("q6k_rep", 1792, [1664], 70, (32, 7, 1)),          # K slices over 13 x 3 tiles
    ("q5k_rep", 2560, [1408], 300, (32, 2, 1)),         # K slices over 11 x 10 tiles
    ("q5k", 1280, [896, 256], 150, (32, 5, 1)),         # raw tier, K slices over 9 x 5 tiles
    # K slices in the grouped order, fewer panels than a group
    ("q5k_rep", 1024, [128], 769, (32, 4, 1)),
    ("q5k", 512, [128], 769, (32, 4, 1)),
    ("q6k_rep", 768, [128], 769, (32, 3, 1)),
    # leftover tiles as K slices, in the narrow last group (of 2)
    ("q5k_rep", 1024, [1664, 1152], 1100, (32, 1, 4)),
    ("q5k", 1280, [2304], 897, (32, 1, 4)),
    # 128-token tiles, whole: 47 / 47 / 55 panels (a last group of 7) x 9 token tiles
    ("q5k_rep", 512, [3072, 2944], 1025, (128, 1, 1)),
    ("q5k", 256, [6016], 1025, (128, 1, 1)),
    ("q6k_rep", 256, [7040], 1025, (128, 1, 1)),
    # 128-token tiles in K slices: 20 (a last group of 4), 3 and 22 (of 6) panels
    ("q5k_rep", 3072, [2560], 1409, (128, 2, 1)),
    ("q5k", 3840, [384], 2049, (128, 5, 1)),
    ("q6k_rep", 3072, [2816], 1100, (128, 2, 1)),
    # 128-token tiles, leftover tiles as K slices in a last group of 2 / 1 panels
    ("q5k_rep", 1024, [2304, 1024], 2500, (128, 1, 4)),
    ("q5k", 512, [7296], 1025, (128, 1, 4)),
]


@pytest.mark.parametrize("fmt,K,Ns,rows,launch", CASES)
def test_every_tile_in_its_place(bq, oracle, fmt, K, Ns, rows, launch):
    import torch
    print(f"tile order {fmt} K={K} Ns={Ns} rows={rows} launch={launch}", flush=True)
    q5 = fmt.startswith("q5k")
    raws = [weights(700 + p + K + n, n, K, "q5k" if q5 else "q6k") for p, n in enumerate(Ns)]
    _, (xq, xd, xs) = acts(711 + rows, rows, K)
    sel = np.array([m for m in range(rows) if launch[0] == 32 or m % 32 in (0, 13, 31) or m == rows - 1])
    sq, sd, ss = xq[sel], xd[sel], xs[sel]
    ws, refs = [], []
    for raw, n in zip(raws, Ns):
        g = dev(raw)
        if fmt == "q5k_rep":
            w144, dm = bq.repack_q5k(g, K, n)
            ws.append(bq.make_weight(g, bq.TYPE_Q5_K, K, n, rep=w144, rep_min=dm))
            r144, rdm = oracle.repack_q5k_144(raw, K)
            refs.append(oracle.gemm_q5k_144(r144, rdm, sq, sd, oracle.fill_xdh(sd, ss), n))
        elif q5:
            ws.append(bq.make_weight(g, bq.TYPE_Q5_K, K, n))
            refs.append(oracle.gemm_q5k(raw, sq, sd, ss))
        else:
            ws.append(bq.make_weight(g, bq.TYPE_Q6_K, K, n, rep=bq.repack_q6k(g, K, n)))
            refs.append(oracle.gemm_q6k(raw, sq, sd))
    ys = [torch.full((rows, n), float("nan"), device="cuda") for n in Ns]
    xdh = torch.zeros((rows, K // 32), dtype=torch.int16, device="cuda")
    bq.gemm_b_fused(ys, ws, rows, dev(xq), dev(xd), dev(xs), xdh)
    torch.cuda.synchronize()
    for p, (y, ref) in enumerate(zip(ys, refs)):
        yh = host(y)
        assert np.isfinite(yh).all()
        check(oracle, yh[sel], ref, what=f"{fmt} part {p}")
