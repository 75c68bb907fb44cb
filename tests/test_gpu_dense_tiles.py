"""The dense op's wide tiles and its split-K kernel at the edges of their tiles and of their
dispatch, against the float64 product of the same quantised operands.

Products are exact and summed in fp32, then one rounding to fp16: half an fp16 ulp of the value
(2^-11) plus the fp32 sums' rounding, which stays below 2^-11 of the largest output at these
sizes: 2^-10 of the largest in all."""
import pytest
import torch

import w4a8_fp8_wmma as W
from w4a8_fp8_wmma import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(M, N, K, asym, seed, dtype=torch.float16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randint(-2**31, 2**31 - 1, (N, K // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    s = (torch.rand((N, K // 128), generator=g, device=DEV) * 0.015 + 0.005).to(torch.float16)
    z = (torch.randint(-2**31, 2**31 - 1, (N // 8, K // 128), generator=g, device=DEV,
                       dtype=torch.int64).to(torch.int32) if asym else None)
    x = torch.randn((M, K), generator=g, device=DEV).to(dtype)
    return x, w, s, z


def _e4m3(b):
    return b.view(torch.float8_e4m3fn).to(torch.float32).double()


def _ref(x, w, s, z):
    q, sc = W.act_quant_fp8(x.to(torch.float16))
    wd = _e4m3(W.dequant_fp8(w, 128, z)) * s.double().repeat_interleave(128, dim=1)
    return (_e4m3(q) @ wd.t()) * sc.double()[:, None]


def _check(x, w, s, z, kernel):
    got = W.mmq_fp8_gemm(x, w, s, kernel=kernel, w_zeros=z).double()
    ref = _ref(x, w, s, z)
    assert float((got - ref).abs().max() / ref.abs().max()) <= 2.0 ** -10


# one row to past each tile's, columns in whole 16s and not (a multiple of 8 with zero-points),
# K of one group, odd numbers of groups, past 16 and past 32 (the tables' chunks)
@pytest.mark.parametrize("M,N,K", [(1, 1000, 128), (17, 136, 384), (33, 264, 2176), (49, 128, 4224),
                                   (64, 520, 2048), (65, 1032, 4352), (129, 256, 6272), (200, 72, 12288)])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("kernel", ["prefill_wmma_ashuffle", "decode_gemv"])
def test_few_tiles(M, N, K, asym, kernel):
    _check(*_case(M, N, K, asym, M + N + K), kernel)


# large grids, ragged at both ends
@pytest.mark.parametrize("M,N,K", [(1090, 4104, 640), (1500, 8200, 384), (2050, 4360, 2304),
                                   (1921, 16328, 256), (4097, 12296, 128)])
@pytest.mark.parametrize("asym", [True, False])
def test_many_tiles(M, N, K, asym):
    _check(*_case(M, N, K, asym, M + N + K), "prefill_wmma_ashuffle")


def _misrounded(M, N, K, asym, rows, kernel="prefill_wmma_ashuffle"):
    """Share of results that are not the float64 value rounded once, and the largest error over the
    largest output. Zero-points 6 .. 10 (around the middle of uniform nibbles)."""
    x, w, s, _ = _case(M, N, K, False, M + N + K)
    if rows == "non-negative":
        x = x.abs()
    z = None
    if asym:
        g = torch.Generator(device=DEV).manual_seed(N)
        v = torch.randint(6, 11, (N // 8, 8, K // 128), generator=g, device=DEV, dtype=torch.int32)
        z = sum(v[:, j] << (4 * j) for j in range(8)).to(torch.int32).contiguous()
    got = W.mmq_fp8_gemm(x, w, s, kernel=kernel, w_zeros=z).double()
    ref = _ref(x, w, s, z)
    return float((got != ref.half().double()).float().mean()), float((got - ref).abs().max() / ref.abs().max())


# The sums' error shows in the results that it moves across a rounding boundary: weights decoded
# to n - z give 1.9 to 2.6% with normal rows and 0.1 to 0.7% with non-negative ones, raw nibbles
# whose zero-point term is taken off afterwards 4.1 to 4.9% and 1.0 to 3.6%.
LIMIT = {"normal": 0.035, "non-negative": 0.008}


# 17 and 33 K groups: past the first and the second scale table, an odd number of groups; rows and
# columns in whole tiles and not. By the rule's costs on 256 compute units: 32 x 64, 64 x 64,
# 64 x 128 (eight waves), 128 x 128 and 256 x 128 tiles
@pytest.mark.parametrize("M,N", [(50, 5000), (200, 4040), (256, 4032), (380, 4088), (1000, 4088), (2000, 4088),
                                 (2048, 4096)])
@pytest.mark.parametrize("K", [2176, 4224])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("rows", ["normal", "non-negative"])
def test_every_tile_past_its_tables(M, N, K, asym, rows):
    share, worst = _misrounded(M, N, K, asym, rows)
    assert share <= LIMIT[rows] and worst <= 2.0 ** -10


# the split-K kernel: 16 to 64 rows a work-group, fewer and more K groups than its waves' loads in
# flight, uneven slices, K of few groups (some waves without any)
@pytest.mark.parametrize("M,N,K", [(9, 520, 5120), (17, 4088, 4224), (40, 1000, 12288), (48, 4096, 1152),
                                   (64, 1032, 8320), (100, 2040, 6144)])
@pytest.mark.parametrize("asym", [True, False])
@pytest.mark.parametrize("rows", ["normal", "non-negative"])
def test_split_k_rounding(M, N, K, asym, rows):
    share, worst = _misrounded(M, N, K, asym, rows)
    assert share <= LIMIT[rows] and worst <= 2.0 ** -10


@pytest.mark.parametrize("rows", ["normal", "non-negative"])
def test_down_projection_of_a_prompt(rows):
    """96 groups: six tables of the largest tile, rows quantised a work-group each."""
    share, worst = _misrounded(2048, 4096, 12288, True, rows)
    assert share <= LIMIT[rows] and worst <= 2.0 ** -10


@pytest.mark.parametrize("M,N,K", [(1, 256, 2048), (9, 512, 4096), (16, 256, 1024), (40, 1024, 2048),
                                   (70, 520, 4352), (300, 1032, 1152)])
def test_bf16_rows_equal_their_fp16_cast(M, N, K):
    x, w, s, z = _case(M, N, K, True, M + K, torch.bfloat16)
    args = (w, s, z, None, None, None, N, K, 128, True, 0, 0)
    a = torch.ops.vllm.w4a8_dense_apply(x, *args)
    b = torch.ops.vllm.w4a8_dense_apply(x.to(torch.float16), *args)
    assert torch.equal(a, b)


@pytest.mark.parametrize("M,N,K", [(17, 12288, 256), (300, 2048, 4096), (600, 4096, 1024)])
def test_gemv_by_name(M, N, K, monkeypatch):
    """The name "decode_gemv" runs the GEMV at any size: the same bits with a workspace, without
    one (the rows then quantised in the kernel) and through the op with its boundary past M."""
    x, w, s, z = _case(M, N, K, True, M + K)
    want = W.mmq_fp8_gemm(x, w, s, kernel="decode_gemv", w_zeros=z)
    bare = torch.empty_like(want)
    _lib.check(_lib.lib.w4a8_mmq_fp8_gemm(
        x.data_ptr(), M, K, w.data_ptr(), s.data_ptr(), z.data_ptr(), N, 128, W._DENSE_KERNELS["decode_gemv"],
        0, bare.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream), "dense")
    monkeypatch.setenv("VLLM_ROCM_W4A8_DECODE_MAX_M", "1000")
    op = torch.ops.vllm.w4a8_dense_apply(x, w, s, z, None, None, None, N, K, 128, True, 0, 0)
    tiles = W.mmq_fp8_gemm(x, w, s, kernel="prefill_wmma_ashuffle", w_zeros=z)
    assert torch.equal(want, bare) and torch.equal(want, op) and not torch.equal(want, tiles)


# no rows: an empty result and no launch, whichever kernel the sizes choose
@pytest.mark.parametrize("N,K", [(256, 1024), (256, 1152), (520, 12288), (12296, 4352)])
@pytest.mark.parametrize("kernel", ["prefill_wmma_ashuffle", "decode_gemv"])
def test_no_rows(N, K, kernel):
    x, w, s, z = _case(0, N, K, True, N + K)
    assert tuple(W.mmq_fp8_gemm(x, w, s, kernel=kernel, w_zeros=z).shape) == (0, N)
