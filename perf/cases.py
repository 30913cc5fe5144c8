"""The work that a user of this package has it do, as measurable cases.

A quantised decoder layer goes through the package at five places, and every case is one of them:

  linear   a front (Quantizer, OnlineHadamard + Quantizer, RMSNorm + Quantizer, or the Hadamard across attention's
           heads + Quantizer) and the Linear4bit layers behind it that share its codes.  `style` says how the program is
           put together: "fused" with this package's fused modules, "modules" with the module-by-module chain of a
           program written for the reference, whose modules all have a counterpart here.
  step     one decode step of the paged int4 cache over `layers` layers: `update` with every layer's new key and value,
           then attention for every layer's query.
  prompt   the keys and values of a batch of prompts, quantised into the pages of the cache.

Sizes are those of the repository's benchmark workloads (hidden widths 4096 / 5120 / 8192, MLP widths 11008 / 13824 /
28672, 8 to 64 heads of 128) plus generic ones; token counts run from one decoded token to 32768 prompt tokens.
"""
import math

import torch

import quarot_amd as quarot
from quarot_amd import nn as qnn
from quarot_amd.transformers.kv_cache import MultiLayerPagedKVCache4Bit, quantize_append_kv_i4

HIDDEN = {4096: 11008, 5120: 13824, 8192: 28672}          # hidden width -> MLP width
HEAD_DIM = 128


def _linear(name, front, tokens, width, out, layers=1, style="fused", fp32=False, bias=False):
    return {"name": name, "kind": "linear", "front": front, "style": style, "tokens": tokens, "in": width, "out": out,
            "layers": layers, "fp32": fp32, "bias": bias}


def listed():
    return [
        # chat with one user: the attention input of a 7B-sized layer for one decoded token (norm, q, k, v) ...
        _linear("token1_norm_qkv_4096", "norm", 1, 4096, 4096, layers=3),
        # ... and the MLP output of the same layer, behind its online Hadamard
        _linear("token1_had_down_11008", "had", 1, 11008, 4096),
        # a small serving batch, 7 sequences, on a 70B-sized MLP input: a token count that fills no tile
        _linear("token7_norm_gateup_8192", "norm", 7, 8192, 28672, layers=2),
        # a larger serving batch on a 13B-sized MLP output
        _linear("token48_had_down_13824", "had", 48, 13824, 5120),
        # a short prompt through a program that keeps the reference's separate modules: RMSNorm, Quantizer, q, k, v
        _linear("prompt333_modules_qkv_4096", "norm", 333, 4096, 4096, layers=3, style="modules"),
        # the benchmark's own workload: 2048 tokens through a 7B-sized down_proj
        _linear("prompt2048_had_down_11008", "had", 2048, 11008, 4096),
        # a prompt of odd length with the Hadamard in fp32, the reference benchmark's second setting, at 70B size
        _linear("prompt1777_fp32had_28672", "had", 1777, 28672, 8192, fp32=True),
        # a batch of prompts at the attention output of a 13B-sized layer: Hadamard across 40 heads, o_proj with a bias
        _linear("prompt8191_heads_o_5120", "heads", 8191, 5120, 5120, bias=True),
        # 16 prompts of 2048 tokens at the MLP input of a 7B-sized layer: the largest batch of the benchmark
        _linear("prompt32768_norm_gateup_4096", "norm", 32768, 4096, 11008, layers=2),
        # decode attention of one long conversation, the reference's attention benchmark: few blocks, all latency
        {"name": "step_1x2048_32heads", "kind": "step", "batch": 1, "length": 2048, "heads": 32, "page": 16, "layers": 8},
        # decode attention of a full serving batch with grouped key-value heads, one odd length
        {"name": "step_32x4001_8heads", "kind": "step", "batch": 32, "length": 4001, "heads": 8, "page": 16, "layers": 4},
        # a batch of prompts of different lengths into the pages of the cache
        {"name": "prompt_cache_12x1500_32heads", "kind": "prompt", "batch": 12, "length": 1500, "heads": 32, "page": 16},
    ]


_MOST_OPS = 2.0 * 32768 * 4096 * 11008 * 2                # the largest listed linear case
_MOST_WEIGHT = 2 * 28672 * 8192                           # and the widest weights


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 5 + ["step"] * 2 + ["prompt"])
    if kind == "step":
        while True:
            case = {"kind": "step", "batch": _log(rng, 1, 64), "length": _log(rng, 64, 16384), "heads": rng.choice([8, 16, 32, 40, 64]),
                    "page": rng.choice([16, 16, 32, 128]), "layers": rng.choice([4, 8])}
            if case["batch"] * (case["length"] + 64) * case["heads"] * case["layers"] <= 32 * 4096 * 8 * 4:
                return case
    if kind == "prompt":
        while True:
            case = {"kind": "prompt", "batch": _log(rng, 1, 32), "length": _log(rng, 16, 8192), "heads": rng.choice([8, 16, 32, 40, 64]),
                    "page": rng.choice([16, 16, 32, 128])}
            if case["batch"] * case["length"] * case["heads"] <= 32 * 4096 * 8:
                return case
    while True:
        tokens = _log(rng, 1, 64) if kind == "decode" else _log(rng, 65, 32768)
        front = rng.choice(["norm", "norm", "had", "had", "quant", "heads"])
        hidden = rng.choice(sorted(HIDDEN))
        mlp = HIDDEN[hidden]
        layers = 1
        if front == "norm":
            width = hidden
            layers, out = rng.choice([(3, hidden), (2, mlp)])
        elif front == "had":
            width, out = rng.choice([(mlp, hidden), (mlp, hidden), (hidden, hidden)])
        elif front == "heads":
            width = out = hidden
        else:                                             # a plain layer: fused qkv or gate_up, or any width at all
            width, out = rng.choice([(hidden, 3 * hidden), (hidden, 2 * mlp), (64 * _log(rng, 16, 448), _log(rng, 512, 28672))])
        style = "modules" if rng.random() < 0.25 else "fused"
        fp32 = front == "had" and rng.random() < 0.3
        case = _linear("", front, tokens, width, out, layers, style, fp32, rng.random() < 0.25)
        del case["name"]
        if 2.0 * tokens * width * out * layers <= _MOST_OPS and width * out * layers <= _MOST_WEIGHT:
            return case


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _activations(gen, tokens, width):
    """fp16, N(0, 1), one channel in a hundred twenty times as large."""
    x = _randn(gen, tokens, width)
    x[:, torch.randperm(width, generator=gen, device="cuda")[:max(1, width // 100)]] *= 20
    return x.half()


def _layer(gen, width, out, bias):
    """A Linear4bit that holds rounded Gaussian weights, as a checkpoint would."""
    with torch.device("cuda"):
        lin = qnn.Linear4bit(width, out, bias=bias).half()
    w = (_randn(gen, out, width) * 0.02).half()
    scales = (w.abs().amax(dim=1, keepdim=True) / 7).half()
    lin.weight, lin.weight_scales = quarot.sym_quant(w, scales), scales
    if bias:
        lin.bias = _randn(gen, out).half()
    return lin


def _prepare_linear(case, gen):
    width, front, fused = case["in"], case["front"], case["style"] == "fused"
    lins = [_layer(gen, width, case["out"], case["bias"]) for _ in range(case["layers"])]
    x = _activations(gen, case["tokens"], width)
    if front == "heads":
        x = x.view(1, case["tokens"], width // HEAD_DIM, HEAD_DIM)          # [batch, tokens, heads, head_dim]
        front_module = qnn.HeadsHadamardQuantizer(width // HEAD_DIM) if fused else qnn.OnlineHadamard(width // HEAD_DIM)
    elif front == "norm":
        front_module = (qnn.RMSNormQuantizer if fused else qnn.RMSNorm)(width)
    else:
        # a layer of its own behind this front: one Sequential from the activations to the output
        chain = [qnn.OnlineHadamard(width, force_fp32=case["fp32"])] if front == "had" else []
        sequential = qnn.Linear4bitSequential if fused else torch.nn.Sequential
        front_module = sequential(*chain, qnn.Quantizer(), lins.pop())
    return {"kind": "linear", "x": x, "front": front_module.cuda(), "lins": lins, "quantizer": qnn.Quantizer(),
            "style": case["style"], "heads": front == "heads"}


def _run_linear(state):
    x = state["x"]
    if not state["lins"]:
        return [state["front"](x)]
    if state["style"] == "fused":
        packed = state["front"](x)
    else:
        if state["heads"]:
            y = state["front"](x.transpose(-1, -2)).transpose(-1, -2)
            y = y.reshape(x.shape[0], x.shape[1], -1).contiguous()
        else:
            y = state["front"](x)
        packed = state["quantizer"](y)
    return [lin(packed) for lin in state["lins"]]


def _vectors(gen, *shape):
    """fp16 keys or values, N(0, 1), one in two hundred fifteen times as large."""
    x = _randn(gen, *shape)
    return torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.005, x * 15, x).half()


def _prepare_step(case, gen):
    batch, length, heads, layers = case["batch"], case["length"], case["heads"], case["layers"]
    cache = MultiLayerPagedKVCache4Bit(batch, case["page"], length + 32, "cuda", layers, heads, HEAD_DIM)
    cache.pages.zero_(), cache.scales.zero_()
    for layer in range(layers):                            # the prompt
        cache.update(_vectors(gen, batch, length - 1, heads, HEAD_DIM), _vectors(gen, batch, length - 1, heads, HEAD_DIM), layer)
    new = [[_vectors(gen, batch, 1, heads, HEAD_DIM) for _ in range(3)] for _ in range(layers)]
    return {"kind": "step", "cache": cache, "first": length - 1, "heads": heads, "new": new}


def _run_step(state):
    cache = state["cache"]
    if cache.length == state["first"] + 32:                # the answer is at its end: the next one continues from the same prompt
        cache.length = state["first"]
    return [cache.update(k, v, layer)(q) for layer, (q, k, v) in enumerate(state["new"])]


def _lengths(case):
    """Prompt lengths around case["length"], from half of it to one and a half times."""
    n, most = case["batch"], case["length"]
    return [max(1, most // 2 + (most * i) // max(1, n - 1)) if n > 1 else most for i in range(n)]


def _prepare_prompt(case, gen):
    heads, page = case["heads"], case["page"]
    lengths = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
    pages = (lengths + page - 1) // page
    total = int(pages.sum())
    start = lambda n: torch.nn.functional.pad(torch.cumsum(n, 0, dtype=torch.int32), (1, 0))
    order = torch.randperm(total, generator=gen, device="cuda").to(torch.int32)
    shape = (int(lengths.sum()), heads, HEAD_DIM)
    return {"kind": "prompt", "k": _vectors(gen, *shape), "v": _vectors(gen, *shape), "seqlens": start(lengths), "specs": {
        "kv_data": torch.zeros(total, 1, 2, heads, page, HEAD_DIM // 2, dtype=torch.uint8, device="cuda"),
        "kv_param": torch.zeros(total, 1, 2, heads, page, 2, dtype=torch.float16, device="cuda"),
        "kv_indptr": start(pages), "kv_indices": order, "last_page_offset": (lengths - 1) % page + 1}}


def _run_prompt(state):
    quantize_append_kv_i4(**state["specs"], k=state["k"], v=state["v"], seqlen_indptr=state["seqlens"], layer_idx=0)
    return [state["specs"]["kv_data"], state["specs"]["kv_param"]]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    return {"linear": _prepare_linear, "step": _prepare_step, "prompt": _prepare_prompt}[case["kind"]](case, gen)


def run(state):
    return {"linear": _run_linear, "step": _run_step, "prompt": _run_prompt}[state["kind"]](state)


def work(case):
    if case["kind"] == "linear":
        m, k, n, layers = case["tokens"], case["in"], case["out"], case["layers"]
        return {"bytes": 2 * m * k + layers * (n * k // 2 + 2 * n + 2 * m * n + (2 * n if case["bias"] else 0)),
                "flops": 2.0 * m * k * n * layers}
    if case["kind"] == "step":
        vectors = case["batch"] * case["heads"]             # 64 bytes of codes and 4 of parameters, for K and for V
        per_layer = vectors * (136 * (case["length"] + 16) + 4 * 2 * HEAD_DIM)
        return {"bytes": case["layers"] * per_layer, "flops": 4.0 * HEAD_DIM * vectors * case["length"] * case["layers"]}
    vectors = 2 * sum(_lengths(case)) * case["heads"]
    return {"bytes": vectors * (2 * HEAD_DIM + 68), "flops": vectors * HEAD_DIM * math.log2(HEAD_DIM)}


def tolerance(case):
    """About four times what each path was seen to differ from itself with its front, its products and its attention in
    float64 on the same inputs."""
    if case["kind"] == "step":                              # seen: 3.6e-4, 2.6e-3
        return {"rel": 1.5e-3, "max": 1e-2}
    if case["kind"] == "prompt":                            # seen: parameters 4e-6, 8.4e-4 (one fp16 step); codes 3.5e-7
        return {"rel": 2e-5, "max": 4e-3, "differ": 2e-6}
    if case["front"] in ("had", "heads") and not case["fp32"]:
        # the transform rounds to fp16 between its two factors: a value one fp16 step away can take the next of 16 codes;
        # seen: 1.2e-2, 0.17
        return {"rel": 2.5e-2, "max": 0.7}
    return {"rel": 1.5e-3, "max": 7e-2}                     # fp16 results of exact integer sums; seen: 3.6e-4, 1.7e-2
