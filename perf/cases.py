"""Workloads of the W4A8 package, as a serving program issues them.

A case is one call (or one replay of a captured decode step) of:

  * ``int4``  - a gated MoE layer with int4 weights of group 128: router plus experts through
    ``moe_forward``, the expert path behind vLLM's MoeWNA16 method through the installed hook,
    or a HIP graph of eight consecutive ``moe_forward`` layers, as an engine captures decode;
  * ``dense`` - one int4 linear layer through ``torch.ops.vllm.w4a8_dense_apply``;
  * ``mxfp4`` - a gpt-oss style MoE layer (E2M1 codes, E8M0 block scales, biases, swigluoai)
    through the installed hook.

Weights are normal values rounded to int4 around their zero-points (mxfp4: uniform codes),
activations are normal, routing is uniform or Zipf(1.1). ``exact`` restates each layer in
float64 with the layer's own rounding points (e4m3 activations, fp16 gate, up and h).
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "rdna4-vllm_amd"))

import w4a8_fp8_wmma as W  # noqa: E402
from w4a8_fp8_wmma import linear, moe_experts  # noqa: E402

linear.register_dense_op()

GROUP = 128
GRAPH_LAYERS = 8
MX_BLOCK = 32


def listed():
    moe = dict(kind="int4", H=2048, I=512, E=256, k=8, zp=True, dtype="bf16", zipf=False)
    big = dict(kind="int4", H=4096, I=1536, E=128, k=8, zp=False, dtype="fp16", zipf=False)
    mx = dict(kind="mxfp4", H=2880, I=2880, E=32, k=4, dtype="bf16")
    return [
        # one user decoding, no graph: the smallest call, where the host and each launch count
        dict(moe, name="int4_decode_t1", entry="forward", T=1),
        # a decode batch replayed from a captured step: eight layers back to back
        dict(moe, name="int4_decode_graph_t32", entry="graph", T=32),
        # decode of the larger experts behind vLLM's hook: symmetric weights, fp16, odd batch
        dict(big, name="int4_hook_t13_h4096", entry="hook", T=13),
        # decode with expert widths of 18 and 7 groups, which the fragment layout does not take
        dict(moe, name="int4_hook_t24_h2304", entry="hook", T=24, H=2304, I=896, E=128),
        # a mixed batch: decoding users and a chunk of somebody's prompt
        dict(moe, name="int4_mixed_t333", entry="forward", T=333),
        # prompt processing with the skewed expert popularity of trained routers
        dict(moe, name="int4_prefill_t4096", entry="forward", T=4096, zipf=True),
        # prompt processing of the larger experts: the largest call
        dict(big, name="int4_prefill_t2048_h4096", entry="forward", T=2048, zp=True, dtype="bf16"),
        # an attention projection while one user decodes
        dict(kind="dense", name="dense_m1", M=1, N=4096, K=4096, zp=True, dtype="fp16"),
        # a wide projection (fused qkv or gate/up) for a decode batch in bf16
        dict(kind="dense", name="dense_m48", M=48, N=12288, K=4096, zp=False, dtype="bf16"),
        # a down projection during prompt processing
        dict(kind="dense", name="dense_m2048", M=2048, N=4096, K=12288, zp=True, dtype="fp16"),
        # gpt-oss decode and prompt processing
        dict(mx, name="mxfp4_decode_t8", T=8),
        dict(mx, name="mxfp4_prefill_t1000", T=1000),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("int4", "int4", "int4", "dense", "dense", "mxfp4"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind == "dense":
        K = GROUP * _log(rng, 8, 96)
        N = 64 * _log(rng, 16, min(192, 4096 * 12288 // K // 64))
        return dict(kind=kind, M=_log(rng, 1, 2048), N=N, K=K, zp=rng.random() < 0.5, dtype=dtype)
    if kind == "mxfp4":
        H, I, E = rng.choice(((2880, 2880, 32), (2880, 2880, 8), (2048, 1024, 32)))
        return dict(kind=kind, H=H, I=I, E=E, k=4, dtype=dtype, T=_log(rng, 1, 1000))
    H, I, E, k = rng.choice(((2048, 512, 256, 8), (2048, 512, 256, 8), (4096, 1536, 128, 8),
                             (2304, 896, 128, 8), (1024, 512, 64, 6), (512, 256, 64, 8)))
    T = _log(rng, 1, 2048 if H == 4096 else 4096)
    entry = rng.choice(("forward", "hook", "graph") if T <= 96 and H == 2048 else ("forward", "hook"))
    if H == 2304:
        entry = "hook"
    return dict(kind=kind, H=H, I=I, E=E, k=k, zp=rng.random() < 0.7, dtype=dtype,
                zipf=rng.random() < 0.5, entry=entry, T=T)


# --------------------------------------------------------------------------- inputs
def _gen(seed, part):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + part)


def _torch_dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float16


def _int4_weight(g, E, N, K, zp):
    """Op-layout words (E, N, K/8), fp16 scales (E, N, G), zero-points as numbers (E, N, G):
    normal weights of standard deviation 2.6 steps, rounded around zero-points of 6 to 10."""
    G = K // GROUP
    z = (torch.randint(6, 11, (E, N, G), generator=g, device="cuda", dtype=torch.int32) if zp
         else torch.full((E, N, G), 8, device="cuda", dtype=torch.int32))
    s = (torch.rand((E, N, G), generator=g, device="cuda") * 0.008 + 0.004).to(torch.float16)
    w = torch.empty((E, N, K // 8), dtype=torch.int32, device="cuda")
    step = max(1, (1 << 26) // (N * K))
    for lo in range(0, E, step):
        hi = min(E, lo + step)
        v = torch.randn((hi - lo, N, G, GROUP), generator=g, device="cuda").mul_(2.6)
        v = v.add_(z[lo:hi, :, :, None]).round_().clamp_(0, 15).to(torch.int32)
        v = v.view(hi - lo, N, K // 8, 8)
        word = v[..., 0].clone()
        for j in range(1, 8):
            word |= v[..., j] << (4 * j)
        w[lo:hi] = word
    return w, s, z


def _pack_zeros(z):
    """Zero-points (E, N, G) -> op layout (E, N/8, G) int32, nibble n % 8 of word n / 8."""
    E, N, G = z.shape
    v = z.view(E, N // 8, 8, G)
    out = v[:, :, 0].clone()
    for j in range(1, 8):
        out |= v[:, :, j] << (4 * j)
    return out.contiguous()


def _zero_bytes(z):
    """Zero-points (E, N, G) -> MoeWNA16 bytes (E, N/2, G), even row in the low nibble."""
    return (z[:, 0::2] | (z[:, 1::2] << 4)).to(torch.uint8).contiguous()


def _tokens(case, seed):
    g = _gen(seed, 3)
    T, E = case["T"], case["E"]
    x = torch.randn((T, case["H"]), generator=g, device="cuda").to(_torch_dtype(case))
    if case.get("zipf"):
        p = 1.0 / torch.arange(1, E + 1, device="cuda", dtype=torch.float64) ** 1.1
        perm = torch.randperm(E, generator=g, device="cuda")
        u = torch.rand((T, E), generator=g, device="cuda", dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
        logits = (torch.log(p / p.sum())[perm] - torch.log(-torch.log(u))).to(torch.float32)
    else:
        logits = torch.randn((T, E), generator=g, device="cuda")
    return x, logits


def _route(logits, k):
    """Softmax, top-k, renormalise, in float64."""
    p, ids = torch.topk(torch.softmax(logits.double(), dim=1), k, dim=1)
    return p / p.sum(dim=1, keepdim=True), ids


class _Quant:
    weight_bits = 4

    def __init__(self, has_zp):
        self.has_zp = has_zp


class _Wna16Method:
    """The part of vLLM's MoeWNA16Method that the hook replaces."""

    def __init__(self, has_zp):
        self.quant_config = _Quant(has_zp)

    def process_weights_after_loading(self, layer):
        pass

    def apply(self, layer, x, topk_weights, topk_ids, shared_experts=None, shared_experts_input=None):
        raise RuntimeError("the stock apply must not run")


class _Mxfp4Method:
    """The part of vLLM's GptOssMxfp4MoEMethod that the hook replaces."""

    def process_weights_after_loading(self, layer):
        raise RuntimeError("the stock load step must not run")

    def apply(self, layer, x, topk_weights, topk_ids, **kw):
        raise RuntimeError("the stock apply must not run")


moe_experts.install_moe_wna16_hooks(_Wna16Method)
moe_experts.install_moe_mxfp4_hooks(_Mxfp4Method)


class _Layer:
    def __init__(self, E, activation, **params):
        self.activation, self.global_num_experts, self.expert_map = activation, E, None
        self.apply_router_weight_on_input = False
        for name, v in params.items():
            setattr(self, name, torch.nn.Parameter(v, requires_grad=False)
                    if isinstance(v, torch.Tensor) else v)


def _int4_layer(case, seed, layer=0):
    g = _gen(seed, 100 + layer)
    E, H, I = case["E"], case["H"], case["I"]
    return _int4_weight(g, E, 2 * I, H, case["zp"]), _int4_weight(g, E, H, I, case["zp"])


def _fragments(case, seed, layer=0):
    (w13, s13, z13), (w2, s2, z2) = _int4_layer(case, seed, layer)
    z13, z2 = (_pack_zeros(z13), _pack_zeros(z2)) if case["zp"] else (None, None)
    if W.fragments_supported(case["H"], case["I"], GROUP):
        w13, w2 = W.repack_fragments(w13, s13, z13), W.repack_fragments(w2, s2, z2)
    return w13, w2, s13, s2, z13, z2


def _mx_weights(case, seed):
    g = _gen(seed, 200)
    E, H, I = case["E"], case["H"], case["I"]

    def codes(*shape):
        return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)

    def exps(*shape):
        return torch.randint(116, 121, shape, generator=g, device="cuda", dtype=torch.uint8)

    def bias(*shape):
        return torch.randn(shape, generator=g, device="cuda").mul_(0.1).to(torch.float16)

    return dict(w13_weight=codes(E, 2 * I, H // 2), w13_weight_scale=exps(E, 2 * I, H // MX_BLOCK),
                w2_weight=codes(E, H, I // 2), w2_weight_scale=exps(E, H, I // MX_BLOCK),
                w13_bias=bias(E, 2 * I), w2_bias=bias(E, H))


def _dense_inputs(case, seed):
    w, s, z = _int4_weight(_gen(seed, 300), 1, case["N"], case["K"], case["zp"])
    x = torch.randn((case["M"], case["K"]), generator=_gen(seed, 3), device="cuda")
    return x.to(_torch_dtype(case)), w[0], s[0], z


def prepare(case, seed):
    if case["kind"] == "dense":
        x, w, s, z = _dense_inputs(case, seed)
        zp = _pack_zeros(z)[0] if case["zp"] else None
        return dict(case=case, x=x, w=w, s=s, z=zp)
    x, logits = _tokens(case, seed)
    if case["kind"] == "mxfp4":
        method, layer = _Mxfp4Method(), _Layer(case["E"], "swigluoai", **_mx_weights(case, seed))
        method.process_weights_after_loading(layer)
        tw, ids = W.fused_topk(x, logits, case["k"], True)
        return dict(case=case, method=method, layer=layer, x=x, tw=tw, ids=ids)
    if case["entry"] == "hook":
        (w13, s13, z13), (w2, s2, z2) = _int4_layer(case, seed)
        p = dict(w13_qweight=w13.view(torch.uint8), w13_scales=s13, w2_qweight=w2.view(torch.uint8),
                 w2_scales=s2, group_size=GROUP)
        if case["zp"]:
            p.update(w13_qzeros=_zero_bytes(z13), w2_qzeros=_zero_bytes(z2))
        method, layer = _Wna16Method(case["zp"]), _Layer(case["E"], "silu", **p)
        method.process_weights_after_loading(layer)
        tw, ids = W.fused_topk(x, logits, case["k"], True)
        return dict(case=case, method=method, layer=layer, x=x, tw=tw, ids=ids)
    state = dict(case=case, x=x, logits=logits, weights=_fragments(case, seed))
    if case["entry"] == "graph":
        layers = [state["weights"]] + [_fragments(case, seed, i) for i in range(1, GRAPH_LAYERS)]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for w in layers:
                W.moe_forward(x, logits, case["k"], *w)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = [W.moe_forward(x, logits, case["k"], *w) for w in layers]
        state.update(weights=layers, graph=graph, outs=outs)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "dense":
        return torch.ops.vllm.w4a8_dense_apply(
            state["x"], state["w"], state["s"], state["z"], None, None, None, case["N"], case["K"],
            GROUP, case["zp"], 0 if case["zp"] else 8, 0)
    if "method" in state:
        return state["method"].apply(state["layer"], state["x"], state["tw"], state["ids"])
    if case["entry"] == "graph":
        state["graph"].replay()
        return state["outs"]
    return W.moe_forward(state["x"], state["logits"], case["k"], *state["weights"])


# --------------------------------------------------------------------------- what a pass needs
def _distinct(case):
    """Experts that the routing touches, expected."""
    E, n = case["E"], case["T"] * case["k"]
    if not case.get("zipf"):
        return E * (1.0 - (1.0 - case["k"] / E) ** case["T"])
    p = [1.0 / i ** 1.1 for i in range(1, E + 1)]
    t = sum(p)
    return sum(1.0 - (1.0 - v / t) ** n for v in p)


def work(case):
    if case["kind"] == "dense":
        M, N, K = case["M"], case["N"], case["K"]
        w = N * K / 2 + N * (K // GROUP) * (2.5 if case["zp"] else 2)
        return dict(bytes=w + 2 * M * (N + K), flops=2.0 * M * N * K)
    T, H, I, E, k = (case[n] for n in ("T", "H", "I", "E", "k"))
    values = 3 * H * I                                     # weights of an expert
    if case["kind"] == "mxfp4":
        expert = values / 2 + values / MX_BLOCK + 2 * (2 * I + H)
    else:
        expert = values / 2 + values / GROUP * (2.5 if case["zp"] else 2)
    layers = GRAPH_LAYERS if case.get("entry") == "graph" else 1
    route = 4 * T * E + 8 * T * k if case.get("entry") in ("forward", "graph") else 8 * T * k
    return dict(bytes=layers * (_distinct(case) * expert + 4 * T * H + route),
                flops=layers * 2.0 * T * k * values)


def tolerance(case):
    if case["kind"] == "dense":
        # exact products, fp32 sums, fp16 results: 2.1e-4 from the float64 layer
        return {"rel": 9e-4}
    # h is rounded to e4m3 between the GEMMs: a last-bit difference of one of its fp16 values
    # moves that value by up to a sixteenth; results are bf16 or fp16: 1.2e-3 to 2.8e-3 from the
    # float64 layer
    return {"rel": 1.2e-2}


# --------------------------------------------------------------------------- float64 restatement
def _quant(x):
    """Rows (fp16) -> e4m3 values and row scales, both float64 (the layer's own rounding)."""
    f = x.to(torch.float16).to(torch.float32)
    amax = f.abs().amax(dim=1, keepdim=True)
    s = (amax / torch.full_like(amax, 448.0)).clamp_min(1e-8)   # a division, not a product
    q = (f * (1.0 / s)).to(torch.float8_e4m3fn)
    return q.to(torch.float32).double(), s.double()


def _half(v):
    """float64 -> fp16 values, as float64."""
    return v.to(torch.float32).to(torch.float16).double()


def _int4_values(w, s, z):
    """One expert's words (N, K/8), scales and zero-points (N, G) -> float64 (N, K)."""
    N = w.shape[0]
    n = torch.stack([(w >> (4 * j)) & 15 for j in range(8)], dim=-1).view(N, -1, GROUP)
    return ((n - z[:, :, None]).double() * s.double()[:, :, None]).view(N, -1)


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _mx_values(w, e):
    """One expert's E2M1 bytes (N, K/2) and E8M0 exponents (N, K/32) -> float64 (N, K)."""
    table = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device=w.device)
    n = torch.stack((w & 15, w >> 4), dim=-1).view(w.shape[0], -1, MX_BLOCK)
    return (table[n.long()] * torch.exp2(e.double() - 127)[:, :, None]).view(w.shape[0], -1)


def _experts(case, x, tw, ids, expert):
    """Sum over a token's experts; expert(e) gives (w13, w2, b13, b2) in float64."""
    a, sa = _quant(x)
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in torch.unique(ids).tolist():
        tok, j = torch.nonzero(ids == e, as_tuple=True)
        w13, w2, b13, b2 = expert(e)
        gu = _half((a[tok] @ w13.t()) * sa[tok])
        if b13 is None:
            gate, up = gu.chunk(2, dim=1)
            h = _half(_half(gate / (1.0 + torch.exp(-gate))) * up)
        else:
            gu = _half(gu + b13)
            gate, up = gu[:, 0::2].clamp_max(7.0), gu[:, 1::2].clamp(-7.0, 7.0)
            h = _half((up + 1.0) * (gate / (1.0 + torch.exp(-1.702 * gate))))
        hq, sh = _quant(h)
        y = (hq @ w2.t()) * sh
        if b2 is not None:
            y = y + b2
        out.index_add_(0, tok, y * tw[tok, j][:, None])
    return out


def exact(case, seed):
    if case["kind"] == "dense":
        x, w, s, z = _dense_inputs(case, seed)
        a, sa = _quant(x)
        return (a @ _int4_values(w, s, z[0]).t()) * sa
    x, logits = _tokens(case, seed)
    tw, ids = _route(logits, case["k"])
    if case["kind"] == "mxfp4":
        m = _mx_weights(case, seed)
        return _experts(case, x, tw, ids, lambda e: (
            _mx_values(m["w13_weight"][e], m["w13_weight_scale"][e]),
            _mx_values(m["w2_weight"][e], m["w2_weight_scale"][e]),
            m["w13_bias"][e].double(), m["w2_bias"][e].double()))
    outs = []
    for i in range(GRAPH_LAYERS if case["entry"] == "graph" else 1):
        (w13, s13, z13), (w2, s2, z2) = _int4_layer(case, seed, i)
        out = _experts(case, x, tw, ids, lambda e: (
            _int4_values(w13[e], s13[e], z13[e]), _int4_values(w2[e], s2[e], z2[e]), None, None))
        outs.append((out, tw, None))
    if case["entry"] == "hook":
        return outs[0][0]
    return outs if case["entry"] == "graph" else outs[0]
