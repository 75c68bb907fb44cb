"""The decode GEMV where its waves do not split K's groups evenly (op layout), against the
float64 product of the same quantised operands.

Products are exact and summed in fp32, then one rounding to fp16: half an fp16 ulp (2^-11) plus
the sums' rounding, below 2^-11 of the largest output at these sizes: 2^-10 of the largest."""
import numpy as np
import pytest
import torch

import bench
import oracle as O
import w4a8_fp8_wmma as W
from w4a8_fp8_wmma import moe_experts

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


def _op(x, w, s, z, ids, block_m, kernel):
    sti, eid, ntp = W.moe_align_block_size(ids, block_m, w.shape[0])
    y = W.mmq_fp8_moe_gemm(x, w, s, sti, eid, ntp, ids.shape[1], block_m, kernel=kernel, w_zeros=z)
    real = (sti < ids.numel()) & (torch.arange(sti.numel(), device=DEV) < ntp)
    return y[real], sti[real].long() // ids.shape[1], eid.repeat_interleave(block_m)[real].long()


@pytest.mark.parametrize("G", [5, 7, 10, 14, 18, 23])
@pytest.mark.parametrize("block_m", [32, 64])
def test_many_rows_in_a_block(G, block_m):
    """Few slots an expert on average, 37 of them with one expert: several passes of 16 rows."""
    E, T, N, K = 32, 37, 72, G * 128
    g = torch.Generator(device=DEV).manual_seed(G + block_m)
    words = lambda *s: torch.randint(-2**31, 2**31 - 1, s, generator=g, device=DEV,
                                     dtype=torch.int64).to(torch.int32)
    w, z = words(E, N, K // 8), words(E, N // 8, G)
    s = (torch.rand((E, N, G), generator=g, device=DEV) * 0.015 + 0.005).to(torch.float16)
    x = torch.randn((T, K), generator=g, device=DEV).to(torch.float16)
    ids = torch.stack([torch.full((T,), 3), torch.randint(4, E, (T,))], 1).to(torch.int32).to(DEV)
    got, tok, e = _op(x, w, s, z, ids, block_m, "gemv")
    q, sc = W.act_quant_fp8(x)
    xd = _e4m3(q) * sc.double()[:, None]
    ref = torch.zeros_like(got, dtype=torch.float64)
    for i in range(E):
        at = (e == i).nonzero()[:, 0]
        wd = _e4m3(W.dequant_fp8(w[i], 128, z[i])) * s[i].double().repeat_interleave(128, 1)
        ref[at] = xd[tok[at]] @ wd.t()
    assert got.shape[0] == 2 * T
    assert float(((got.double() - ref).abs().amax(1) / ref.abs().amax(1)).max()) <= 2.0 ** -10


@pytest.mark.parametrize("T,block_m", [(17, 32), (17, 64), (130, 16)])
def test_many_slots_an_expert_run_the_tiles(T, block_m):
    """Past 8 slots an expert (64 in 16-row blocks) both names run the tiles: the same bits."""
    E, N, G = 4, 264, 7
    g = torch.Generator(device=DEV).manual_seed(T + block_m)
    words = lambda *s: torch.randint(-2**31, 2**31 - 1, s, generator=g, device=DEV,
                                     dtype=torch.int64).to(torch.int32)
    w, z = words(E, N, G * 16), words(E, N // 8, G)
    s = (torch.rand((E, N, G), generator=g, device=DEV) * 0.015 + 0.005).to(torch.float16)
    x = torch.randn((T, G * 128), generator=g, device=DEV).to(torch.float16)
    ids = torch.rand((T, E), generator=g, device=DEV).argsort(1)[:, :2].to(torch.int32).contiguous()
    assert torch.equal(_op(x, w, s, z, ids, block_m, "gemv")[0], _op(x, w, s, z, ids, block_m, "wmma")[0])
    few = ids[:4].contiguous()   # 2 slots an expert: the GEMV
    assert not torch.equal(_op(x[:4], w, s, z, few, block_m, "gemv")[0], _op(x[:4], w, s, z, few, block_m, "wmma")[0])


# each split in gemm1 (gate and up, SiLU) and in gemm2 (slot outputs); one to four tiles a
# work-group in gemm1, up to eight in gemm2
@pytest.mark.parametrize("H,I", [(640, 128), (896, 640), (1152, 896), (1280, 1152), (1408, 1280), (1664, 1408),
                                 (1920, 1792), (2176, 2176), (2304, 2560), (2688, 2688), (3072, 3072)])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("T,E", [(3, 4), (40, 64)])
def test_decode_layer_equals_composition(H, I, asym, T, E):
    """A decode layer on the op layout against gemm (checked above), silu_and_mul, gemm and
    gather-reduce. The composition rounds y to fp16 (half an ulp: 2^-11 of each term) and both
    round the output (2^-11 each): within 2^-9 of the largest output; a wrong gate, up, scale or
    zero-point is off by its own size."""
    g = torch.Generator(device=DEV).manual_seed(H + I + T + asym)
    words = lambda *s: torch.randint(-2**31, 2**31 - 1, s, generator=g, device=DEV,
                                     dtype=torch.int64).to(torch.int32)
    scales = lambda *s: (torch.rand(s, generator=g, device=DEV) * 0.015 + 0.005).to(torch.float16)
    w13, w2 = words(E, 2 * I, H // 8), words(E, H, I // 8)
    s13, s2 = scales(E, 2 * I, H // 128), scales(E, H, I // 128)
    z13, z2 = (words(E, 2 * I // 8, H // 128), words(E, H // 8, I // 128)) if asym else (None, None)
    x = (torch.randn((T, H), generator=g, device=DEV) * 0.1).to(torch.float16)
    ids = torch.rand((T, E), generator=g, device=DEV).argsort(1)[:, :2].to(torch.int32).contiguous()
    tw = torch.rand((T, 2), generator=g, device=DEV)
    out = W.moe_apply(x, w13, w2, s13, s2, z13, z2, tw, ids).float()
    ref = moe_experts._run_unfused(x, w13, w2, s13, s2, z13, z2, tw.reshape(-1), ids, 2, E, None,
                                   "gemv", False, None, None, 16).float()
    assert torch.isfinite(out).all() and float((out - ref).abs().max()) <= 2.0 ** -9 * float(ref.abs().max())


@pytest.mark.parametrize("H,I", [(2304, 896), (640, 1152), (1664, 2816)])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("T", [3, 24])
def test_decode_layer_vs_oracle(H, I, asym, T):
    """A decode layer with uneven K groups in both GEMMs: SiLU and slot outputs, the layer's bar."""
    ws = bench.make_weights(dict(T=T, H=H, E=8, k=2, I=I, g=128, routing="uniform"), H + T, DEV)
    z13, z2 = (ws["z13"], ws["z2"]) if asym else (None, None)
    x, logits = bench.make_inputs(dict(T=T, H=H, E=8, k=2, I=I, g=128, routing="uniform"), I + T, DEV)
    tw, ids = W.fused_topk(None, logits, 2, True)
    out = W.moe_apply(x, ws["w13"], ws["w2"], ws["s13"], ws["s2"], z13, z2, tw, ids)
    n = lambda t: None if t is None else t.cpu().numpy()
    ref = O.moe_layer(n(x.float()), n(ws["w13"]), n(ws["s13"]), n(z13), n(ws["w2"]), n(ws["s2"]),
                      n(z2), n(tw), n(ids), 128, round_y_fp16=False)
    assert np.abs(n(out.float()) - ref).max() <= 1e-2 * np.abs(ref).max()


def test_bounds_of_the_tiles_stay():
    """Where the tiles refused a call of these sizes the GEMV refuses it too: weights of 2 GiB an
    expert (its offsets are 32-bit), blocks of 8 rows."""
    K = 5 * 128
    x = torch.zeros((16, K), dtype=torch.float16, device=DEV)
    route = [torch.zeros(n, dtype=torch.int32, device=DEV) for n in (16, 2, 1)]

    def call(N, block_m):
        w = torch.empty((1, N, K // 8), dtype=torch.int32, device=DEV)
        s = torch.empty((1, N, 5), dtype=torch.float16, device=DEV)
        return W.mmq_fp8_moe_gemm(x, w, s, route[0], route[1][:16 // block_m].contiguous(), route[2], 1, block_m,
                                  kernel="gemv")

    assert tuple(call(64, 16).shape) == (16, 64)
    for N, block_m in ((64, 8), (2 ** 32 // K + 8, 16)):
        with pytest.raises(RuntimeError, match="multiple of 16|2 GiB"):
            call(N, block_m)
