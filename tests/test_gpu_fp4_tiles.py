"""E2M1 tiles with groups of 32: the block-scaled MFMA form (scales that are powers of two), the
general form (any fp16 scale) and the whole mxfp4 layer in one call.

The tiles and the scalar kernel sum the same exact products in fp32, in different orders, and
round once to fp16: results within one fp16 ulp of each other, so within 2^-10 of the largest
one, plus the sums' own difference (4e-6 of the results against float64, below 2^-13 of the
largest): TOL."""
import numpy as np
import pytest
import torch

import oracle as O
import w4a8_fp8_wmma as W
from w4a8_fp8_wmma import moe_experts

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 2.0 ** -10 + 2.0 ** -13


def _dev(*arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in arrays]


def _maxrel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _scales(r, kind, E, N, G):
    s = 2.0 ** r.integers(-14, 3, (E, N, G))
    if kind == "late":        # one scale of the last group of one row is no power of two
        s[E // 2, N // 3, G - 1] = 0.3
    if kind == "first":       # ... of the first group of one row of each expert
        s[:, N // 2, 0] = 0.0117
    if kind == "all":         # every row of half the experts: no ring, the general form at once
        s[::2] *= 1.0 + 0.5 * r.random((s[::2].shape[0], N, G))
    if kind == "zero":        # zero and subnormal scales
        s[0, :, G // 2] = 0.0
        s[E - 1, 1, 0] = 2.0 ** -20
    return s.astype(np.float16)


# (N, K): one step, a partial step, K past four steps, gpt-oss's 22.5 steps, an odd number of
# groups; columns in whole fragments and not
@pytest.mark.parametrize("N,K", [(64, 128), (256, 160), (200, 608), (320, 2880), (136, 1120)])
@pytest.mark.parametrize("block_m", [16, 32, 64, 128])
@pytest.mark.parametrize("kind", ["powers", "late", "first", "zero", "all"])
def test_tiles_match_scalar(N, K, block_m, kind):
    T, E, k = 45, 4, 2
    r = np.random.default_rng(N + K + block_m + len(kind))
    w = r.integers(-2**31, 2**31, (E, N, K // 8), dtype=np.int64).astype(np.int32)
    s = _scales(r, kind, E, N, K // 32)
    x = r.standard_normal((T, K)).astype(np.float16)
    ids = np.stack([r.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    sti, eid, ntp = O.moe_align(ids, block_m, E)
    args = _dev(x, w, s, sti, eid, ntp)
    real = np.nonzero(sti[:int(ntp[0])] < T * k)[0]
    got, ref = (W.mmq_fp8_moe_gemm(*args, k, block_m, kernel=kern, weight_is_e2m1=True)
                .float().cpu().numpy()[real] for kern in ("wmma", "scalar"))
    assert np.isfinite(got).all() and _maxrel(got, ref) <= TOL
    half = N // 2
    if half % 16 == 0:   # gate and up halves, SiLU in the epilogue, against the op by op form
        h = W.mmq_fp8_moe_gemm1_silu(*args, k, block_m, weight_is_e2m1=True)
        full = W.mmq_fp8_moe_gemm(*args, k, block_m, kernel="wmma", weight_is_e2m1=True)
        want = torch.empty_like(h)
        W.silu_and_mul(want, full)
        # a column's form does not depend on the tile it is in
        assert np.array_equal(h.float().cpu().numpy()[real], want.float().cpu().numpy()[real])


@pytest.mark.parametrize("H,I,T", [(2880, 2880, 1), (2880, 2880, 33), (2880, 2880, 170), (128, 160, 5),
                                   (1024, 544, 70),
                                   # the last and first sizes of the shared align and row launch
                                   (160, 128, 256), (160, 128, 257), (4096, 128, 9), (4128, 128, 9)])
@pytest.mark.parametrize("act,bias,dtype", [("swigluoai", True, torch.bfloat16),
                                            ("silu", True, torch.float16),
                                            ("swigluoai", False, torch.float32)])
def test_layer_call_equals_composition(H, I, T, act, bias, dtype):
    """One native call against the op by op composition on the same tiles, bit for bit, with
    an expert map that drops some slots."""
    E, n_global, k = 6, 8, 4
    r = np.random.default_rng(H + I + T)
    w13, w2 = (r.integers(-2**31, 2**31, sh, dtype=np.int64).astype(np.int32)
               for sh in ((E, 2 * I, H // 8), (E, H, I // 8)))
    s13, s2 = (2.0 ** r.integers(-11, -6, sh) for sh in ((E, 2 * I, H // 32), (E, H, I // 32)))
    b13, b2 = (r.standard_normal(sh).astype(np.float32) * 0.1 for sh in ((E, 2 * I), (E, H)))
    ids = np.stack([r.permutation(n_global)[:k] for _ in range(T)]).astype(np.int32)
    tw = r.random((T, k)).astype(np.float32)
    emap = np.array([3, -1, 0, 5, 1, -1, 2, 4], np.int32)
    w13, w2, s13, s2, b13, b2, ids, tw, emap = _dev(
        w13, w2, s13.astype(np.float16), s2.astype(np.float16), b13, b2, ids, tw, emap)
    if not bias:
        b13 = b2 = None
    x = torch.from_numpy(r.standard_normal((T, H)).astype(np.float32)).to(DEV).to(dtype)
    out_dtype = torch.bfloat16 if dtype == torch.bfloat16 else torch.float16
    got = moe_experts._run_grouped_moe(x, w13, w2, s13, s2, None, None, tw, ids, act, n_global,
                                       emap, False, "wmma", out_dtype=out_dtype,
                                       weight_is_e2m1=True, w1_bias=b13, w2_bias=b2)
    ref = moe_experts._run_unfused(x.to(torch.float16), w13, w2, s13, s2, None, None,
                                   tw.reshape(-1), ids, k, n_global, emap, "wmma", True, b13, b2,
                                   64, act).to(out_dtype)
    assert torch.isfinite(got.float()).all()
    assert torch.equal(got, ref)


@pytest.mark.parametrize("H,block_m", [(512, 16), (2880, 16), (2880, 32), (2880, 64), (2880, 128)])
@pytest.mark.parametrize("kind", ["powers", "all"])
@pytest.mark.parametrize("rows", ["normal", "non-negative"])
def test_sums_against_float64(H, block_m, kind, rows):
    """The fp32 sums themselves (scatter output, one slot a token): the block-scaled form adds a
    step's four groups and all steps inside the MFMA. Both forms, and one MFMA and a fold per
    group before, measure 3.9 to 4.2e-6 (2-norm); raising a group's weight or losing a bit of the
    sum shows at once. Bound: 6e-6."""
    N, E, T = 320, 4, 60
    r = np.random.default_rng(H + block_m)
    w = r.integers(-2**31, 2**31, (E, N, H // 8), dtype=np.int64).astype(np.int32)
    s = (2.0 ** r.integers(-12, -5, (E, N, H // 32)) * (1.0 if kind == "powers" else 1.0 + 0.5 * r.random((E, N, H // 32))))
    x = r.standard_normal((T, H))
    ids = r.integers(0, E, (T, 1)).astype(np.int32)
    sti, eid, ntp = O.moe_align(ids, block_m, E)
    real = sti < T
    xp = np.zeros((len(sti), H))
    xp[real] = (np.abs(x) if rows == "non-negative" else x)[sti[real]]
    w, s, xp, sti_d, eid, ntp = _dev(w, s.astype(np.float16), xp.astype(np.float16), sti, eid, ntp)
    out = torch.zeros((T, N), device=DEV)
    W.mmq_fp8_moe_gemm_scatter(xp, w, s, sti_d, eid, ntp, torch.ones(T, device=DEV), out, 1, block_m,
                               weight_is_e2m1=True)
    q, sc = W.act_quant_fp8(xp)
    xd = q.view(torch.float8_e4m3fn).float().double() * sc.double()[:, None]
    code = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=DEV)
    nib = torch.stack([(w >> (4 * j)) & 15 for j in range(8)], -1).reshape(E, N, H).long()
    wd = torch.where(nib >= 8, -code[nib % 8], code[nib % 8]) * s.double().repeat_interleave(32, 2)
    ref = torch.zeros((T, N), dtype=torch.float64, device=DEV)
    for p in np.nonzero(real)[0]:
        t = int(sti[p])
        ref[t] = wd[int(ids[t, 0])] @ xd[p]
    assert float((out.double() - ref).norm() / ref.norm()) <= 6e-6
