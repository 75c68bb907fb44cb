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
    a large value at the end and a zero row among them."""
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
    assert bool(((q & 0x7F) == 0x7F)[~keep].all())   # NaN stays NaN


@pytest.mark.parametrize("K", [4224, 8192, 16384])
def test_infinite_rows_and_bf16(K):
    """An infinity (in bf16 also a value past fp16's range, which the cast makes one) gives an
    infinite scale: finite values quantise to 0, the infinity to NaN. bf16 rows enter through the
    dense op; with K = 4224 and more they take a work-group each."""
    x = torch.randn((4, K), generator=torch.Generator(device=DEV).manual_seed(K), device=DEV)
    x[1, K - 3] = float("inf")
    x[2, 7] = -float("inf")
    x[3, 4100] = 1e6
    q, s = W.act_quant_fp8(x.half())
    assert torch.isinf(s[1:]).all() and torch.isfinite(s[0])
    bad = torch.isinf(x.half())
    assert bool(((q[1:] & 0x7F) == 0x7F)[bad[1:]].all()) and bool(((q[1:] & 0x7F) == 0)[~bad[1:]].all())
    g = torch.Generator(device=DEV).manual_seed(K)
    w = torch.randint(-2**31, 2**31 - 1, (64, K // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    sc = torch.full((64, K // 128), 0.01, device=DEV, dtype=torch.float16)
    args = (w, sc, None, None, None, None, 64, K, 128, False, 8, 0)
    b = x.to(torch.bfloat16)
    got = torch.ops.vllm.w4a8_dense_apply(b, *args)
    want = torch.ops.vllm.w4a8_dense_apply(b.half(), *args)
    assert torch.isfinite(got[0]).all() and torch.isnan(got[1:]).all()
    assert torch.equal(got[0], want[0]) and torch.isnan(want[1:]).all()
