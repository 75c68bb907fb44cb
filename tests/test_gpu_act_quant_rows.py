"""Act-quant of rows past 4096 values (a work-group a row) against the formula, byte for byte."""
import pytest
import torch

import w4a8_fp8_wmma as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("K", [4104, 8192, 16384, 16392])
@pytest.mark.parametrize("rows", [1, 5])
def test_long_rows_quantise_as_short_ones(K, rows):
    """Rows past 4096 values take a work-group each: the bytes and scales of the formula, a NaN,
    an infinity and a zero row among them."""
    g = torch.Generator(device=DEV).manual_seed(K + rows)
    x = torch.randn((rows, K), generator=g, device=DEV).to(torch.float16)
    if rows > 4:
        x[1] = 0
        x[2, K - 1] = 300.0
        x[3, 4100] = float("nan")
    q, s = W.act_quant_fp8(x)
    f = x.float()
    amax = torch.nan_to_num(f.abs(), nan=0.0).amax(dim=1)
    want = (amax / torch.full_like(amax, 448.0)).clamp_min(1e-8)
    assert torch.equal(s, want)
    y = f * (1.0 / want)[:, None]
    keep = ~torch.isnan(y)
    assert torch.equal(q[keep], y.to(torch.float8_e4m3fn).view(torch.uint8)[keep])
