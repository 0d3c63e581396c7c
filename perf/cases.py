"""What a program that serves a quantized model asks of this framework, as measurable cases.

A case is one layer or block of such a model at one token count, called through the
package's public layer surface:

  linear  ``MxLinearMethod.apply``: MXFP8, MXFP6 (E2M3 or E3M2) or block-FP8 weights, bf16 in and out
  mlp     residual + RMSNorm -> gate_up projection -> SwiGLU -> down projection, MXFP8 weights
          (``ops.norm_mx_gate_up`` and ``swiglu_mxfp8_down``), the residual sum returned beside it
  moe     ``Mxfp6Experts.apply_router``: routing, both grouped GEMMs and the weighted combine
          of an MXFP6 mixture of experts, from router logits

The token counts are those of decode batches (1 to 64), of small and chunked prefills (up to
4096) and what lies between; decode cases with ``"graph"`` replay one captured call, as a
serving loop does after its warmup, the others are plain calls.  The weights are in the
checkpoint formats, made from the seed by plain torch arithmetic, so that ``exact`` can make
them again without this package.
"""
from __future__ import annotations

import math

import torch

from __graft_entry__ import load_package

EPS = 1e-6
FP6 = {"mxfp6_e2m3": (2, 3, 1, 2), "mxfp6_e3m2": (3, 2, 3, 4)}  # code, mantissa bits, bias, emax
_capture_stream = None


def listed():
    return [
        # decode, batch 16, an attention-sized projection: the smallest call, launch latency and little else
        dict(name="decode_mxfp8_16", kind="linear", fmt="mxfp8", m=16, n=2048, k=2048, bias=False, graph=True),
        # the same layer family called eagerly for one sequence, with a bias: host and launch cost included
        dict(name="eager_mxfp8_1", kind="linear", fmt="mxfp8", m=1, n=4608, k=2048, bias=True, graph=False),
        # decode of a single sequence through a whole MLP block
        dict(name="decode_mlp_1", kind="mlp", m=1, h=2560, i=9216, graph=True),
        # decode at a batch size between the smallest and a prefill
        dict(name="decode_mlp_48", kind="mlp", m=48, h=2560, i=9216, graph=True),
        # decode through the widest W6A8 layer, an odd batch
        dict(name="decode_mxfp6_27", kind="linear", fmt="mxfp6_e3m2", m=27, n=17408, k=5120, bias=False, graph=True),
        # a short prompt through the block-FP8 gate_up layer
        dict(name="prefill_block_512", kind="linear", fmt="block_fp8", m=512, n=18432, k=2560, bias=False, graph=False),
        # a chunk of prefill through the block-FP8 layer, ragged row count
        dict(name="prefill_block_1777", kind="linear", fmt="block_fp8", m=1777, n=18432, k=2560, bias=False,
             graph=False),
        # a ragged prompt through a W6A8 layer whose K is an odd number of 128-blocks
        dict(name="prefill_mxfp6_333", kind="linear", fmt="mxfp6_e2m3", m=333, n=5120, k=2688, bias=True, graph=False),
        # the largest dense call: a long prefill chunk through the widest W6A8 layer
        dict(name="prefill_mxfp6_4096", kind="linear", fmt="mxfp6_e2m3", m=4096, n=17408, k=5120, bias=False,
             graph=False),
        # a prefill chunk through the MLP block
        dict(name="prefill_mlp_2048", kind="mlp", m=2048, h=2560, i=9216, graph=False),
        # mixture of experts at a decode batch: every expert's weights for a few rows each
        dict(name="decode_moe_64", kind="moe", fmt="mxfp6_e3m2", m=64, h=2048, i=512, e=256, topk=8, graph=True),
        # mixture of experts on a prefill chunk
        dict(name="prefill_moe_2048", kind="moe", fmt="mxfp6_e2m3", m=2048, h=2048, i=512, e=256, topk=8,
             graph=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, q):
    return max(lo, min(hi, _log(rng, lo, hi) // q * q))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "mlp", "mlp", "moe"])
    m = _log(rng, 1, 4096)
    graph = m <= 64 and rng.random() < 0.7
    if kind == "moe":
        return dict(kind=kind, fmt=rng.choice(list(FP6)), m=min(m, 2048), h=_multiple(rng, 1024, 2048, 128),
                    i=_multiple(rng, 256, 512, 128), e=rng.choice([64, 128, 256]), topk=rng.choice([4, 8]), graph=graph)
    if kind == "mlp":
        return dict(kind=kind, m=m, h=_multiple(rng, 1024, 3072, 128), i=_multiple(rng, 2048, 9216, 128), graph=graph)
    fmt = rng.choice(["mxfp8", "block_fp8"] + list(FP6))
    n = _multiple(rng, 512, 17408, 8 if fmt in FP6 else 128)
    return dict(kind=kind, fmt=fmt, m=m, n=n, k=_multiple(rng, 1024, 5120 if n > 9216 else 9216, 128),
                bias=rng.random() < 0.3, graph=graph)


# ------------------------------------------------------------------ inputs, from the seed alone


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _activations(g, m, k):
    """bf16 N(0, 1) with one channel in a hundred twenty times larger, as activations have."""
    x = _randn(g, m, k)
    x[:, torch.randperm(k, generator=g, device="cuda")[: max(1, k // 100)]] *= 20
    return x.bfloat16()


def _mx_weight(g, shape, fmt, std):
    """Checkpoint tensors of an MX weight: (codes, E8M0 scales), one scale per 32 along the last axis."""
    w = _randn(g, *shape, std=std).view(*shape[:-1], -1, 32)
    emax = 8 if fmt == "mxfp8" else FP6[fmt][3]
    e = torch.frexp(w.abs().amax(-1, keepdim=True).clamp_min(1e-20))[1] - 1 - emax
    scale = (e + 127).squeeze(-1).to(torch.uint8)
    v = torch.ldexp(w, -e).view(*shape)
    if fmt == "mxfp8":
        return v.clamp(-448, 448).to(torch.float8_e4m3fn), scale
    table = _fp6_values(fmt)[:32]
    mids = ((table[1:] + table[:-1]) / 2).float()
    codes = torch.bucketize(v.abs(), mids) + 32 * (v < 0)
    c = codes.to(torch.int32).view(*shape[:-1], -1, 4)
    bits = c[..., 0] | c[..., 1] << 6 | c[..., 2] << 12 | c[..., 3] << 18
    packed = torch.stack([bits & 255, bits >> 8 & 255, bits >> 16 & 255], -1).to(torch.uint8)
    return packed.view(*shape[:-1], shape[-1] * 3 // 4), scale


def _fp6_values(fmt):
    """The 64 values of an FP6 format by code (the sign is bit 5), in 64 bits."""
    _, mb, bias, _ = FP6[fmt]
    c = torch.arange(32, device="cuda")
    e, f = c >> mb, (c & ((1 << mb) - 1)).double() / (1 << mb)
    v = torch.where(e == 0, f * 2.0 ** (1 - bias), (1 + f) * torch.exp2((e - bias).double()))
    return torch.cat([v, -v])


def _block_weight(g, n, k, std):
    """Checkpoint tensors of a block-FP8 weight: E4M3 codes [N, K] and fp32 scales per 128 x 128."""
    w = _randn(g, n, k, std=std).view(n // 128, 128, k // 128, 128)
    s = w.abs().amax(dim=(1, 3)) / 448.0
    return (w / s[:, None, :, None]).view(n, k).clamp(-448, 448).to(torch.float8_e4m3fn), s.contiguous()


def _inputs(case, seed):
    g, m = _generator(seed), case["m"]
    if case["kind"] == "linear":
        n, k, fmt = case["n"], case["k"], case["fmt"]
        w, s = _block_weight(g, n, k, 0.02) if fmt == "block_fp8" else _mx_weight(g, (n, k), fmt, 0.02)
        return dict(x=_activations(g, m, k), w=w, s=s, bias=_randn(g, n).bfloat16() if case["bias"] else None)
    h, i = case["h"], case["i"]
    if case["kind"] == "mlp":
        w1, s1 = _mx_weight(g, (2 * i, h), "mxfp8", 0.02)
        w2, s2 = _mx_weight(g, (h, i), "mxfp8", 0.02)
        return dict(x=_activations(g, m, h), res=_randn(g, m, h).bfloat16(), norm=_randn(g, h, std=0.1).bfloat16(),
                    w1=w1, s1=s1, w2=w2, s2=s2)
    w1, s1 = _mx_weight(g, (case["e"], 2 * i, h), case["fmt"], 0.015)
    w2, s2 = _mx_weight(g, (case["e"], h, i), case["fmt"], 0.015)
    return dict(x=_randn(g, m, h).bfloat16(), logits=_randn(g, m, case["e"]), w1=w1, s1=s1, w2=w2, s2=s2)


# ------------------------------------------------------------------ the framework's calls


def _linear_layer(mx, key, n, k, w, s):
    method, layer = mx.MxLinearMethod(key), torch.nn.Module()
    method.create_weights(layer, k, [n], k, n, torch.bfloat16, device="cuda")
    layer.weight.weight_loader(layer.weight, w)
    scale = layer.weight_scale_inv if hasattr(layer, "weight_scale_inv") else layer.weight_scale
    scale.weight_loader(scale, s)
    method.process_weights_after_loading(layer)
    return method, layer


def _program(case, d):
    """The call that a user's program makes on each pass, as a function without arguments."""
    mx = load_package()
    if case["kind"] == "linear":
        key = {"mxfp8": mx.linear.MXFP8_STATIC, "mxfp6_e2m3": mx.linear.MXFP6_E2M3_STATIC,
               "mxfp6_e3m2": mx.linear.MXFP6_E3M2_STATIC, "block_fp8": mx.linear.FP8_BLOCK128}[case["fmt"]]
        method, layer = _linear_layer(mx, key, case["n"], case["k"], d["w"], d["s"])
        return lambda: method.apply(layer, d["x"], d["bias"])
    if case["kind"] == "mlp":
        h, i = case["h"], case["i"]
        _, gate_up = _linear_layer(mx, mx.linear.MXFP8_STATIC, 2 * i, h, d["w1"], d["s1"])
        _, down = _linear_layer(mx, mx.linear.MXFP8_STATIC, h, i, d["w2"], d["s2"])

        def mlp():
            mid, summed = mx.ops.norm_mx_gate_up(d["x"], d["res"], d["norm"], EPS, gate_up.weight,
                                                 gate_up.weight_scale, 2 * i)
            return mx.swiglu_mxfp8_down(mid, down), summed

        return mlp
    experts = mx.Mxfp6Experts(fmt=FP6[case["fmt"]][0])
    w1, w2 = experts.process_weights_after_loading(d["w1"], d["s1"], d["w2"], d["s2"])

    def moe():
        out = torch.empty_like(d["x"])
        experts.apply_router(out, d["x"], w1, w2, d["logits"], case["topk"])
        return out

    return moe


def prepare(case, seed):
    global _capture_stream
    d = _inputs(case, seed)
    call = _program(case, d)
    for name in ("w", "s", "w1", "s1", "w2", "s2"):  # the layers hold their own copies
        d.pop(name, None)
    if not case["graph"]:
        return dict(call=call)
    if _capture_stream is None:  # a program captures on one stream of its own
        _capture_stream = torch.cuda.Stream()
    stream = _capture_stream
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call()
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = call()
    return dict(graph=graph, out=out, call=call)  # the call holds the tensors that the graph reads


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ------------------------------------------------------------------ what a pass cannot do without


def _weight_bytes(n, k, fmt):
    if fmt == "block_fp8":
        return n * k + n * k // 4096
    return n * k * (8 if fmt == "mxfp8" else 6) // 8 + n * k // 32


def work(case):
    m = case["m"]
    if case["kind"] == "linear":
        n, k = case["n"], case["k"]
        return dict(bytes=_weight_bytes(n, k, case["fmt"]) + 2 * m * k + 2 * m * n + 2 * n * case["bias"],
                    flops=2 * m * n * k)
    h, i = case["h"], case["i"]
    if case["kind"] == "mlp":
        return dict(bytes=_weight_bytes(3 * i, h, "mxfp8") + 4 * 2 * m * h + 2 * h, flops=6 * m * h * i)
    # each expert that some token is routed to (uniform routing: the expected share) reads its weights once
    hit = case["e"] * (1 - (1 - case["topk"] / case["e"]) ** m)
    return dict(bytes=int(hit * _weight_bytes(3 * i, h, case["fmt"])) + 4 * m * h + 4 * m * case["e"],
                flops=6 * m * case["topk"] * h * i)


def tolerance(case):
    # bf16 results of fp32 sums, four times what the path measured against ``exact``: a linear layer is off by its
    # one bf16 rounding (1.7e-3, with a bias two: 2.3e-3); in the blocks (up to 3.0e-3) a sum next to a rounding
    # boundary moves the bf16 value between the two projections and with it an 8-bit code
    if case["kind"] == "linear":
        return dict(rel=9e-3 if case["bias"] else 7e-3, max=0.03)
    return dict(rel=1.2e-2, max=0.1)


# ------------------------------------------------------------------ the same in 64 bits, by plain torch


def _dequant_mx(codes, scale, fmt):
    if fmt == "mxfp8":
        v = codes.double()
    else:
        b = codes.view(*codes.shape[:-1], -1, 3).int()
        bits = b[..., 0] | b[..., 1] << 8 | b[..., 2] << 16
        c = torch.stack([bits & 63, bits >> 6 & 63, bits >> 12 & 63, bits >> 18 & 63], -1)
        v = _fp6_values(fmt)[c.long()].view(*codes.shape[:-1], -1)
    s = torch.exp2(scale.double() - 127)
    return (v.view(*scale.shape, 32) * s.unsqueeze(-1)).view(v.shape)


def _quant_mx(x, rule):
    """The values that the dynamic MXFP8 quantization of bf16 ``x`` stands for, in 64 bits."""
    b = x.view(x.shape[0], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    if rule == "floor_carry175":  # exponent of the amax, carried up from 1.75 on
        bits = amax.view(torch.int16).int()
        e = ((bits + 32 & 0xFF80) >> 7) - 8 - 127
    else:  # ceil_div448
        f, e = torch.frexp((amax.float() / 448.0).clamp_min(1e-30))
        e = e - (f == 0.5).int()
    scale = torch.exp2(e.double())
    codes = (b.double() / scale).float().to(torch.float8_e4m3fn)
    return (codes.double() * scale).view(x.shape)


def _quant_block(x):
    b = x.float().view(x.shape[0], -1, 128)
    s = b.abs().amax(-1, keepdim=True).clamp_min(1e-10) / 448.0
    return ((b / s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s.double()).view(x.shape)


def _swiglu(mid):
    g, u = mid.float().chunk(2, -1)
    return ((g / (1 + torch.exp(-g))).bfloat16().float() * u).bfloat16()


def exact(case, seed):
    d = _inputs(case, seed)
    x = d["x"]
    if case["kind"] == "linear":
        if case["fmt"] == "block_fp8":
            s = d["s"].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
            y = _quant_block(x) @ (d["w"].double() * s).t()
        else:
            y = _quant_mx(x, "floor_carry175") @ _dequant_mx(d["w"], d["s"], case["fmt"]).t()
        return y if d["bias"] is None else y + d["bias"].double()
    if case["kind"] == "mlp":
        v = x.double() + d["res"].double()
        y = (v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * (1 + d["norm"].double())).bfloat16()
        mid = (_quant_mx(y, "ceil_div448") @ _dequant_mx(d["w1"], d["s1"], "mxfp8").t()).bfloat16()
        return _quant_mx(_swiglu(mid), "ceil_div448") @ _dequant_mx(d["w2"], d["s2"], "mxfp8").t(), v
    topk = case["topk"]
    p, ids = torch.softmax(d["logits"].double(), -1).topk(topk, -1)
    p = p / p.sum(-1, keepdim=True)
    a, out = _quant_mx(x, "floor_carry175"), torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in range(case["e"]):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if not len(t):
            continue
        mid = (a[t] @ _dequant_mx(d["w1"][e], d["s1"][e], case["fmt"]).t()).bfloat16()
        y = (_quant_mx(_swiglu(mid), "ceil_div448") @ _dequant_mx(d["w2"][e], d["s2"][e], case["fmt"]).t()).bfloat16()
        out.index_add_(0, t, y.double() * p[t, slot].unsqueeze(-1))
    return out
