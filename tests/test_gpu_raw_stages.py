"""The raw Q5_K prefill GEMM's staging (bq_gemm.hip k_mmq_q5k_raw) at the sizes
where it can go wrong: the fewest stages, K slices that start at an odd stage
(the second half of a super-block), token tiles of one row, an odd count of
stages left in a slice, both tile heights.  Against the oracle, with the raw
tier's tolerance (helpers.check).  The launch each case is there for is checked
without a GPU in test_mmq_plan.py."""
import pytest

from helpers import acts, check, dev, host, weights

pytestmark = pytest.mark.gpu

CASES = [
    # K, N, rows, launch (token-tile height, K slices, slices per leftover tile)
    (256, 128, 97, (32, 1, 1)),       # two stages, one weight tile, a last token tile of one row
    (256, 3072, 2049, (128, 1, 1)),   # 128-token tiles, two stages, a last token tile of one row
    (768, 7168, 513, (32, 1, 1)),     # six stages whole, a last token tile of one row
    (512, 7680, 385, (128, 1, 1)),    # 128-token tiles, four stages whole, a last token tile of one row
    (1792, 1280, 129, (32, 5, 1)),    # K slices of 32-token tiles
    (2304, 2560, 640, (32, 1, 1)),    # 18 stages whole
    (2304, 8320, 97, (128, 6, 1)),    # 128-token tiles of 97 rows, six slices of three stages
    (2816, 384, 128, (32, 8, 1)),     # 22 stages in as many slices as a launch may take
]


@pytest.mark.parametrize("K,N,rows,launch", CASES)
def test_raw_stages(bq, oracle, K, N, rows, launch):
    import torch
    print(f"raw stages K={K} N={N} rows={rows} launch={launch}", flush=True)
    raw = weights(900 + K + N, N, K, "q5k")
    _, (xq, xd, xs) = acts(911 + rows, rows, K)
    w = bq.make_weight(dev(raw), bq.TYPE_Q5_K, K, N)
    y = torch.full((rows, N), float("nan"), device="cuda")
    xdh = torch.zeros((rows, K // 32), dtype=torch.int16, device="cuda")
    bq.gemm_b_fused([y], [w], rows, dev(xq), dev(xd), dev(xs), xdh)
    torch.cuda.synchronize()
    check(oracle, host(y), oracle.gemm_q5k(raw, xq, xd, xs), what="raw")
