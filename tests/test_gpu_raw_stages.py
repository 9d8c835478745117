"""The raw Q5_K prefill GEMM's staging (bq_gemm.hip k_mmq_q5k_raw) at the sizes
where it can go wrong: the fewest stages, K slices that start at an odd stage
(the second half of a super-block), token tiles of one row, an odd count of
stages left in a slice, both tile heights.  Against the oracle, with the raw
tier's tolerance (helpers.check)."""
import pytest

from helpers import acts, check, dev, host, weights

pytestmark = pytest.mark.gpu

CASES = [
    # K, N, rows
    (256, 128, 97),       # two stages, one weight tile, a last token tile of one row
    (256, 3072, 2049),    # 128-token tiles, two stages, a last token tile of one row
    (768, 7168, 513),     # 128-token tiles, whole
    (1792, 1280, 129),    # K slices of 32-token tiles
    (2304, 2560, 640),    # 18 stages in K slices of 128-token tiles
    (2816, 384, 128),     # 22 stages in as many slices as the scratch allows
]


@pytest.mark.parametrize("K,N,rows", CASES)
def test_raw_stages(bq, oracle, K, N, rows):
    import torch
    print(f"raw stages K={K} N={N} rows={rows}", flush=True)
    raw = weights(900 + K + N, N, K, "q5k")
    _, (xq, xd, xs) = acts(911 + rows, rows, K)
    w = bq.make_weight(dev(raw), bq.TYPE_Q5_K, K, N)
    y = torch.full((rows, N), float("nan"), device="cuda")
    xdh = torch.zeros((rows, K // 32), dtype=torch.int16, device="cuda")
    bq.gemm_b_fused([y], [w], rows, dev(xq), dev(xd), dev(xs), xdh)
    torch.cuda.synchronize()
    check(oracle, host(y), oracle.gemm_q5k(raw, xq, xd, xs), what="raw")
