"""Performance cases of the weight-quantized linear path: the calls a quantized model
makes while it decodes and while it reads a prompt, through the entry points that
generated modules and Linnet programs use (`linnet_amd.torch.generated`,
`.quantized`, `.nf4`) and one whole decode step (`linnet_amd.llama.Int4Llama`).

The layers are those of an 8B-class decoder (hidden 4096, MLP 14336, q|k|v joined to
6144, gate|up to 28672), a wide FP8 layer (8192 -> 28672) and a mixture of 32 experts
of 2880 (top 4), in every weight format of `std.quant`. `listed()` holds one case of
each use, `draw()` spreads over the same uses' sizes, row counts, groups and types.
Weights are N(0, 0.02) quantized here in plain torch, activations N(0, 1) with a few
larger channels, as norm outputs have.
"""

from __future__ import annotations

import math

import torch

from linnet_amd.llama import Int4Llama
from linnet_amd.torch import generated, kernels, nf4, quantized

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
NF4_VALUES = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
              -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
              0.2461123019456863, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
              0.7229568362236023, 1.0]
FP4_VALUES = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]
HIDDEN, HEADS, KV_HEADS, FFN, VOCAB, LAYERS = 4096, 32, 8, 14336, 128256, 2


def listed():
    return [
        # One token through an attention output projection: the smallest call of a decode step.
        dict(name="int4_one_token", kind="int4", rows=1, k=4096, n=4096, group=128, dtype="bf16", bias=False),
        # A decode batch of 16 through an up projection; groups of 64, f16 and a bias, as GPTQ checkpoints have them.
        dict(name="int4_batch16_group64", kind="int4", rows=16, k=4096, n=14336, group=64, dtype="f16", bias=True),
        # A short prompt (or a chunk of one) through a joined q|k|v projection; ragged in its rows.
        dict(name="int4_short_prompt", kind="int4", rows=200, k=4096, n=6144, group=128, dtype="bf16", bias=False),
        # A long prompt through an up projection.
        dict(name="int4_prompt", kind="int4", rows=2048, k=4096, n=14336, group=128, dtype="bf16", bias=False),
        # Weight-only FP8 for a small decode batch of a wide layer.
        dict(name="fp8_batch8", kind="w8", format="fp8", rows=8, k=8192, n=28672, group=0, dtype="bf16"),
        # Weight-only int8 with a scale per 128 inputs for a decode batch of 24.
        dict(name="int8_group_batch24", kind="w8", format="int8_group", rows=24, k=4096, n=14336, group=128, dtype="bf16"),
        # int8 x int8 (rows rounded per token) for a batch of 128 sequences or a short prompt.
        dict(name="int8_rounded_128", kind="w8a8", format="int8", rows=128, k=4096, n=14336, dtype="bf16"),
        # FP8 x FP8 for a long prompt of the wide layer.
        dict(name="fp8_rounded_prompt", kind="w8a8", format="fp8", rows=4096, k=8192, n=28672, dtype="bf16"),
        # FP8 x FP8 with 128 x 128 block scales for a prompt; ragged in its rows.
        dict(name="fp8_block_prompt", kind="w8a8", format="fp8_block", rows=777, k=4096, n=14336, dtype="bf16"),
        # NF4 (QLoRA) for a small decode batch.
        dict(name="nf4_batch6", kind="nf4", rows=6, k=4096, n=14336, block=64, dtype="bf16", bias=False),
        # A mixture's gate|up experts for a decode batch of 32 tokens, top 4 of 32.
        dict(name="mxfp4_batch32", kind="mxfp4", form="shared", rows=32, top=4, experts=32, k=2880, n=5760, dtype="bf16"),
        # A whole decode step of one sequence (two layers and the head), replayed from a HIP graph.
        dict(name="llama_step", kind="llama", rows=1, context=1024),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _out(rng, most):
    """Output features: a layer's, or anything in its range; two in three a multiple of 64."""
    n = rng.choice([4096, 6144, 14336, 28672]) if rng.random() < 0.3 else _log(rng, 1024, most)
    n = min(n, most)
    return n // 64 * 64 if rng.random() < 2 / 3 else n


def _inputs(rng, step, most):
    k = rng.choice([4096, 14336]) if rng.random() < 0.4 else _log(rng, 1024, most)
    return max(step, min(k, most) // step * step)


def draw(rng):
    kind = rng.choice(["int4", "int4", "int4_prompt", "w8", "w8", "w8a8", "w8a8", "nf4", "nf4", "mxfp4", "mxfp4", "llama"])
    dtype = "bf16" if rng.random() < 0.7 else "f16"
    if kind == "int4":
        group = rng.choice([128, 128, 64, 32])
        return dict(kind="int4", rows=_log(rng, 1, 64), k=_inputs(rng, 128, 14336), n=_out(rng, 28672), group=group,
                    dtype=dtype, bias=rng.random() < 0.3)
    if kind == "int4_prompt":
        k, n = _inputs(rng, 128, 14336), _out(rng, 28672)
        rows = max(65, min(_log(rng, 65, 2048), int(1.2e11 / k / n)))
        return dict(kind="int4", rows=rows, k=k, n=n, group=rng.choice([128, 128, 64, 32]), dtype=dtype,
                    bias=rng.random() < 0.3)
    if kind == "w8":
        form = rng.choice(["fp8", "int8", "int8_group", "fp8_block"])
        k, n = _inputs(rng, 128, 14336), _out(rng, 28672)
        if form == "fp8_block":
            n = max(128, n // 128 * 128)
        group = {"fp8": 0, "int8": 0, "int8_group": rng.choice([64, 128]), "fp8_block": 128}[form]
        return dict(kind="w8", format=form, rows=_log(rng, 1, 64), k=k, n=n, group=group, dtype=dtype)
    if kind == "w8a8":
        form = rng.choice(["fp8", "int8", "fp8_block"])
        k, n = _inputs(rng, 128, 14336), _out(rng, 28672)
        if form == "fp8_block":
            n = max(128, n // 128 * 128)
        rows = max(33, min(_log(rng, 33, 4096), int(2.4e11 / k / n)))
        return dict(kind="w8a8", format=form, rows=rows, k=k, n=n, dtype=dtype)
    if kind == "nf4":
        return dict(kind="nf4", rows=_log(rng, 1, 256), k=_inputs(rng, 64, 14336), n=_out(rng, 28672), block=64,
                    dtype=dtype, bias=rng.random() < 0.3)
    if kind == "mxfp4":
        experts = rng.choice([8, 16, 32])
        return dict(kind="mxfp4", form=rng.choice(["shared", "combine"]), rows=_log(rng, 1, 64), top=rng.choice([2, 4]),
                    experts=experts, k=_log(rng, 1024, 2880) // 32 * 32, n=_log(rng, 1024, 5760), dtype=dtype)
    return dict(kind="llama", rows=_log(rng, 1, 64), context=_log(rng, 64, 2048))


# ------------------------------------------------------------------ inputs, as plain tensors


def _generator(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + salt)


def _activations(g, rows, k, dtype):
    x = torch.randn(rows, k, generator=g, device="cuda")
    wide = torch.randint(0, k, (max(1, k // 512),), generator=g, device="cuda")
    x[:, wide] *= 6.0
    return x.to(dtype)


def _quantize4(w, group):
    """(packed [n, k/group, group/2], scale f32, zero), round to nearest: the checkpoint tools' 4-bit formula."""
    n, k = w.shape
    w = w.view(n, k // group, group)
    low, high = w.amin(-1), w.amax(-1)
    scale = (high - low) / 15.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    zero = torch.round(-low / scale).clamp(0, 15)
    q = (torch.round(w / scale[..., None]) + zero[..., None]).clamp(0, 15).to(torch.uint8)
    return q[..., 0::2] | (q[..., 1::2] << 4), scale, zero.to(torch.uint8)


def _weight(g, n, k):
    return torch.randn(n, k, generator=g, device="cuda").mul_(0.02)


def _int4_tensors(case, seed):
    g = _generator(seed, 1)
    dtype = DTYPES[case["dtype"]]
    packed, scale, zero = _quantize4(_weight(g, case["n"], case["k"]), case["group"])
    x = _activations(g, case["rows"], case["k"], dtype)
    bias = torch.randn(case["n"], generator=g, device="cuda").to(dtype) if case["bias"] else None
    return x, packed, scale.to(dtype), zero, bias


def _byte_tensors(case, seed):
    g = _generator(seed, 2)
    n, k, form = case["n"], case["k"], case["format"]
    w = _weight(g, n, k)
    if form == "int8_group":
        w = w.view(n, k // case["group"], case["group"])
        scale = w.abs().amax(-1) / 127.0
        weight = torch.round(w / scale[..., None]).clamp(-127, 127).to(torch.int8).view(n, k)
    elif form == "int8":
        scale = w.abs().amax(-1) / 127.0
        weight = torch.round(w / scale[:, None]).clamp(-127, 127).to(torch.int8)
    elif form == "fp8":
        scale = w.abs().amax(-1) / 448.0
        weight = (w / scale[:, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    else:
        w = w.view(n // 128, 128, k // 128, 128)
        scale = w.abs().amax((1, 3)) / 448.0
        weight = (w / scale[:, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8).view(n, k)
    return _activations(g, case["rows"], k, DTYPES[case["dtype"]]), weight, scale


def _nf4_tensors(case, seed):
    g = _generator(seed, 3)
    n, k, block = case["n"], case["k"], case["block"]
    dtype = DTYPES[case["dtype"]]
    w = _weight(g, n, k).view(n, k // block, block)
    absmax = w.abs().amax(-1)
    levels = torch.tensor(NF4_VALUES, device="cuda")
    q = torch.bucketize(w / absmax[..., None], (levels[1:] + levels[:-1]) / 2).to(torch.uint8).view(n, k)
    x = _activations(g, case["rows"], k, dtype)
    bias = torch.randn(n, generator=g, device="cuda").to(dtype) if case["bias"] else None
    return x, q[:, 0::2] | (q[:, 1::2] << 4), absmax, bias


def _mxfp4_tensors(case, seed):
    g = _generator(seed, 4)
    e, n, k, rows, top = case["experts"], case["n"], case["k"], case["rows"], case["top"]
    dtype = DTYPES[case["dtype"]]
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda")
    blocks = torch.empty(e, n, k // 32, 16, dtype=torch.uint8, device="cuda")
    for i in range(e):
        w = torch.randn(n, k // 32, 32, generator=g, device="cuda").mul_(2.0)
        q = torch.bucketize(w.abs(), edges).to(torch.uint8) | ((w < 0).to(torch.uint8) << 3)
        blocks[i] = q[..., 0::2] | (q[..., 1::2] << 4)
    scales = torch.randint(118, 123, (e, n, k // 32), generator=g, device="cuda").to(torch.uint8)
    # A router's choice: some experts are chosen more often than others.
    logits = torch.randn(rows, e, generator=g, device="cuda") + 0.5 * torch.randn(e, generator=g, device="cuda")
    weights, experts = logits.topk(top, dim=-1)
    if case["form"] == "shared":
        x = _activations(g, rows, k, dtype)
    else:
        x = _activations(g, rows * top, k, dtype).view(rows, top, k)
    return x, blocks, scales, experts, torch.softmax(weights, -1).to(dtype)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "int4":
        x, packed, scale, zero, bias = _int4_tensors(case, seed)
        return dict(kind=kind, x=x, packed=generated._int4_pack(packed, scale, zero), bias=bias, raw=packed, scale=scale,
                    zero=zero)
    if kind in ("w8", "w8a8"):
        x, weight, scale = _byte_tensors(case, seed)
        form, rounded = case["format"], int(kind == "w8a8")
        if form == "int8_group":
            operands, linear = quantized.int8_group_operands(weight, scale), quantized.int8_group_linear
        elif form == "int8":
            operands, linear = quantized.int8_operands(weight, scale, rounded), quantized.int8_linear
        elif form == "fp8":
            operands, linear = quantized.fp8_operands(weight, scale, rounded), quantized.fp8_linear
        else:
            operands, linear = quantized.fp8_block_operands(weight, scale, rounded), quantized.fp8_block_linear
        return dict(kind=kind, x=x, operands=operands, linear=linear)
    if kind == "nf4":
        x, codes, absmax, bias = _nf4_tensors(case, seed)
        return dict(kind=kind, x=x, codes=codes, absmax=absmax, bias=bias, block=case["block"])
    if kind == "mxfp4":
        x, blocks, scales, experts, weights = _mxfp4_tensors(case, seed)
        return dict(kind=kind, x=x, blocks=blocks, scales=scales, experts=experts,
                    weights=weights if case["form"] == "combine" else None)
    # A decoder serving `rows` sequences: its step recorded once, as a serving loop records it.
    model = Int4Llama(torch, kernels, torch.device("cuda"), layers=LAYERS, hidden=HIDDEN, heads=HEADS, kv_heads=KV_HEADS,
                      ffn=FFN, vocab=VOCAB, ctx=case["context"], batch=case["rows"], seed=int(seed))
    x = _llama_input(case, seed)
    model.step(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = model.step(x)
    return dict(kind=kind, model=model, x=x, graph=graph, logits=logits)


def _llama_input(case, seed):
    return torch.randn(case["rows"], HIDDEN, generator=_generator(seed, 5), device="cuda").mul_(0.5).to(torch.bfloat16)


def run(state):
    kind = state["kind"]
    if kind == "int4":
        return generated._int4_linear(state["x"], state["packed"], state["bias"], state["raw"], state["scale"], state["zero"])
    if kind in ("w8", "w8a8"):
        return state["linear"](state["x"], state["operands"], None)
    if kind == "nf4":
        return nf4.linear_nf4(state["x"], state["codes"], state["absmax"], state["bias"], state["block"])
    if kind == "mxfp4":
        return generated._mxfp4_grouped(state["x"], state["blocks"], state["scales"], state["experts"], state["weights"])
    state["graph"].replay()
    return dict(logits=state["logits"], keys=state["model"].kt, values=state["model"].vc)


# ------------------------------------------------------------------ what the path cannot do without


def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind == "llama":
        qkv = HIDDEN + 2 * KV_HEADS * (HIDDEN // HEADS)
        params = LAYERS * HIDDEN * (qkv + HIDDEN + 3 * FFN) + VOCAB * HIDDEN
        cache = LAYERS * rows * case["context"] * 2 * KV_HEADS * (HIDDEN // HEADS)
        flops = 2 * rows * params + 2 * 2 * cache * (HEADS // KV_HEADS)
        return {"bytes": params * (0.5 + 3 / 128) + cache * 2 + rows * (HIDDEN + VOCAB) * 2, "flops": flops}
    k, n = case["k"], case["n"]
    if kind == "mxfp4":
        pairs = rows * case["top"]
        distinct = case["experts"] * (1 - (1 - case["top"] / case["experts"]) ** rows)
        x = rows if case["form"] == "shared" else pairs
        y = pairs if case["form"] == "shared" else rows
        return {"bytes": distinct * n * k * 17 / 32 + (x * k + y * n) * 2 + pairs * 8, "flops": 2 * pairs * n * k}
    if kind == "int4":
        weight = n * k / 2 + n * (k / case["group"]) * 3
    elif kind == "nf4":
        weight = n * k / 2 + n * (k / case["block"]) * 4
    else:
        scales = {"fp8": n, "int8": n, "fp8_block": n * k / 128 / 128}.get(case["format"])
        weight = n * k + 4 * (n * k / case["group"] if scales is None else scales)
    return {"bytes": weight + rows * (k + n) * 2 + (2 * n if case.get("bias") else 0), "flops": 2 * rows * n * k}


def tolerance(case):
    """About four times what two correct implementations differ by: measured against the same product with the
    weight widened in x's type and multiplied by torch, 2.3e-3 to 3.4e-3 in bf16 and 2.8e-4 to 3.8e-4 in f16 (the
    rounding of the widened weight and of the result), 1e-3 in f16 where the rows are rounded to FP8 (quotients on
    a tie of E4M3). The step's logits are 8e-3 from the 64-bit ones: one rounding of every activation between."""
    if case["kind"] == "llama":
        return {"rel": 2e-2}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 4e-3 if case["kind"] == "w8a8" and case["format"] != "int8" else 1.5e-3}


# ------------------------------------------------------------------ the same in 64 bits


def _codes4(packed):
    return torch.stack([packed & 15, packed >> 4], dim=-1).flatten(-2)


def _int4_weight(packed, scale, zero):
    q = _codes4(packed).double() - zero.double()[..., None]
    return (q * scale.double()[..., None]).flatten(1)


def _nf4_weight(codes, absmax):
    w = torch.tensor(NF4_VALUES, dtype=torch.float64, device="cuda")[_codes4(codes).int()]
    return (w.view(*absmax.shape, -1) * absmax.double()[..., None]).flatten(1)


def _rounded(x, form):
    """The rows as the 8-bit product reads them: rounded to 8 bits with a scale a row (or a 128-input block)."""
    rows, k = x.shape
    x = x.float().view(rows, -1, 128) if form == "fp8_block" else x.float()
    most = 127.0 if form == "int8" else 448.0
    scale = x.abs().amax(-1, keepdim=True).clamp(min=1e-12) / most
    v = x / scale
    if form == "int8":
        q = torch.trunc(v + torch.where(v >= 0, 0.5, -0.5)).clamp(-127, 127)
    else:
        q = v.clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * scale.double()).reshape(rows, k)


def _byte_weight(case, weight, scale):
    n, k = weight.shape
    form = case["format"]
    w = weight.double() if form.startswith("int8") else weight.view(torch.float8_e4m3fn).double()
    if form == "int8_group":
        return (w.view(n, -1, case["group"]) * scale.double()[..., None]).view(n, k)
    if form == "fp8_block":
        return (w.view(n // 128, 128, k // 128, 128) * scale.double()[:, None, :, None]).view(n, k)
    return w * scale.double()[:, None]


def _mxfp4_exact(case, seed):
    x, blocks, scales, experts, weights = _mxfp4_tensors(case, seed)
    rows, top = experts.shape
    xs = (x[:, None, :].expand(rows, top, -1) if x.dim() == 2 else x).double()
    y = torch.zeros(rows, top, case["n"], dtype=torch.float64, device="cuda")
    values = torch.tensor(FP4_VALUES, dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        at = (experts == e).nonzero(as_tuple=True)
        if at[0].numel():
            w = values[_codes4(blocks[e]).int()] * torch.exp2(scales[e].double() - 127)[..., None]
            y[at] = xs[at] @ w.flatten(1).t()
    return y if case["form"] == "shared" else (y * weights.double()[..., None]).sum(1)


def _llama_exact(case, seed):
    """The decode step in 64 bits: weights and caches drawn as the model draws them."""
    rows, ctx, hd = case["rows"], case["context"], HIDDEN // HEADS
    g = torch.Generator(device="cuda").manual_seed(int(seed))

    def linear(n, k):
        packed, scale, zero = _quantize4(torch.randn(n, k, generator=g, device="cuda") * 0.02, 128)
        return packed, scale.to(torch.bfloat16), zero

    def norm():
        return (1 + 0.1 * torch.randn(HIDDEN, generator=g, device="cuda")).double()

    kv = KV_HEADS * hd
    layers = [dict(q=linear(HIDDEN, HIDDEN), k=linear(kv, HIDDEN), v=linear(kv, HIDDEN), o=linear(HIDDEN, HIDDEN),
                   gate=linear(FFN, HIDDEN), up=linear(FFN, HIDDEN), down=linear(HIDDEN, FFN), n1=norm(), n2=norm())
              for _ in range(LAYERS)]
    last, head = norm(), linear(VOCAB, HIDDEN)
    cap = (ctx + 1 + 3) // 4 * 4
    keys = [torch.randn(rows, KV_HEADS, hd, cap, generator=g, device="cuda").to(torch.bfloat16) for _ in range(LAYERS)]
    values = [torch.randn(rows, KV_HEADS, cap, hd, generator=g, device="cuda").to(torch.bfloat16) for _ in range(LAYERS)]
    inv = 1.0 / (500000.0 ** (torch.arange(0, hd, 2, device="cuda", dtype=torch.float32) / hd))
    cos, sin = torch.cos(ctx * inv).double(), torch.sin(ctx * inv).double()

    def rms(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w

    def rope(t):
        a, b = t[..., : hd // 2], t[..., hd // 2 :]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    def times(x, w):
        return x @ _int4_weight(*w).t()

    x = _llama_input(case, seed).double()
    for p, kt, vc in zip(layers, keys, values):
        h = rms(x, p["n1"])
        q = rope(times(h, p["q"]).view(rows, HEADS, hd)).view(rows, KV_HEADS, HEADS // KV_HEADS, hd)
        k = rope(times(h, p["k"]).view(rows, KV_HEADS, hd))
        v = times(h, p["v"]).view(rows, KV_HEADS, hd)
        kt = torch.cat([kt[..., :ctx].double(), k[..., None]], dim=-1)
        vc = torch.cat([vc[:, :, :ctx].double(), v[:, :, None]], dim=2)
        att = torch.softmax(q @ kt * hd ** -0.5, dim=-1) @ vc
        x = x + times(att.reshape(rows, HIDDEN), p["o"])
        h = rms(x, p["n2"])
        x = x + times(torch.nn.functional.silu(times(h, p["gate"])) * times(h, p["up"]), p["down"])
    return dict(logits=times(rms(x, last), head), keys=[None] * LAYERS, values=[None] * LAYERS)


def exact(case, seed):
    kind = case["kind"]
    if kind == "int4":
        x, packed, scale, zero, bias = _int4_tensors(case, seed)
        weight = _int4_weight(packed, scale, zero)
    elif kind in ("w8", "w8a8"):
        x, weight, scale = _byte_tensors(case, seed)
        bias, weight = None, _byte_weight(case, weight, scale)
        x = _rounded(x, case["format"]) if kind == "w8a8" else x
    elif kind == "nf4":
        x, codes, absmax, bias = _nf4_tensors(case, seed)
        weight = _nf4_weight(codes, absmax)
    elif kind == "mxfp4":
        return _mxfp4_exact(case, seed)
    else:
        return _llama_exact(case, seed)
    y = x.double() @ weight.t()
    return y if bias is None else y + bias.double()
