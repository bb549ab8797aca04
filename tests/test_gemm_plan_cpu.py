"""The GEMM's choice of a tile, at products that a wrong choice slows: the plan
for 256 CUs (what a device-less process reckons with), bf16 datapath."""
import pytest

import mxenc

BF16, F32 = mxenc.MX_BF16, mxenc.MX_F32
PAIR = "lds_128x128x64_w64x64_ns2_persistent"  # two 128 x 128 tiles to a CU


@pytest.mark.parametrize("M,K,N,cdt,res,plan", [
    # shallow products: 7-35 % longer on 128 x 256 or 256 x 256 tiles
    (14, 128, 5120, BF16, 0, PAIR),
    (300, 128, 768, F32, 1, PAIR),
    (1500, 192, 768, BF16, 0, PAIR),
    (19000, 192, 64, BF16, 0, PAIR),
    (33000, 320, 384, BF16, 0, PAIR),
    (19000, 384, 384, BF16, 0, PAIR),
    (33000, 448, 1344, BF16, 0, "lds_256x192x32_w64x96_ns4_persistent"),
    # W is read once per row of tiles: 60 us on 64 x 64 ones for 47 and 52
    (1065, 3072, 3840, F32, 1, "lds_128x128x64_w64x64_ns2_persistent"),
    # as small as a tile gets where each has a CU
    (19, 384, 1152, BF16, 0, "lds_64x64x128_w32x32_ns3_mfma16_persistent"),
])
def test_plan(M, K, N, cdt, res, plan):
    assert mxenc.lib().mx_gemm_plan_for(M, N, K, cdt, res, 0).decode() == plan
