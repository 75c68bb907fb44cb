"""The decode GEMV where its waves do not split K's groups evenly (op layout), against the
float64 product of the same quantised operands.

Products are exact and summed in fp32, then one rounding to fp16: half an fp16 ulp (2^-11) plus
the sums' rounding, below 2^-11 of the largest output at these sizes: 2^-10 of the largest."""
import pytest
import torch

import w4a8_fp8_wmma as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _e4m3(b):
    return b.view(torch.float8_e4m3fn).to(torch.float32).double()


# every number of groups outside the even splits, with a last wave that has some, one or none;
# columns past a tile, row blocks with more real rows than one pass takes
@pytest.mark.parametrize("G", [5, 7, 9, 10, 11, 13, 14, 15, 17, 18, 19, 20, 21, 22, 23, 24])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("T,N,block_m", [(1, 48, 16), (5, 136, 16), (37, 40, 64)])
def test_uneven_groups(G, asym, T, N, block_m):
    E, k, K = 4, 2, G * 128
    g = torch.Generator(device=DEV).manual_seed(1000 * G + T + N + asym)
    words = lambda *s: torch.randint(-2**31, 2**31 - 1, s, generator=g, device=DEV,
                                     dtype=torch.int64).to(torch.int32)
    w = words(E, N, K // 8)
    s = (torch.rand((E, N, G), generator=g, device=DEV) * 0.015 + 0.005).to(torch.float16)
    z = words(E, N // 8, G) if asym else None
    x = torch.randn((T, K), generator=g, device=DEV).to(torch.float16)
    ids = torch.rand((T, E), generator=g, device=DEV).argsort(1)[:, :k].to(torch.int32).contiguous()
    sti, eid, ntp = W.moe_align_block_size(ids, block_m, E)
    got = W.mmq_fp8_moe_gemm(x, w, s, sti, eid, ntp, k, block_m, kernel="gemv", w_zeros=z).double()
    q, sc = W.act_quant_fp8(x)
    xd = _e4m3(q) * sc.double()[:, None]
    rows = 0
    for p in range(int(ntp[0])):
        slot, e = int(sti[p]), int(eid[p // block_m])
        if slot >= T * k:
            continue
        wd = _e4m3(W.dequant_fp8(w[e], 128, z[e] if asym else None)) * s[e].double().repeat_interleave(128, 1)
        ref = wd @ xd[slot // k]
        assert float((got[p] - ref).abs().max() / ref.abs().max()) <= 2.0 ** -10
        rows += 1
    assert rows == T * k
