"""The work whose speed is measured: products of whole transformer layers, LM
heads, an encoder block and a whole decode step, through the package's public
entry points (charlotte_amd.matmul), on one GPU.

Weights are made on the GPU in the device layout (the streams that
charlotte_hip_matmul_weight_wrap takes) with the distributions of
charlotte_amd.synthetic: Q4_0 and Q4_1 d = fp16(|N| 0.02), Q8_0 d = fp16(|N|
0.0005), Q6_K d = fp16(|N| 0.001) with int8 scales -64..63, codes uniform;
F32, F16 and BF16 weights N(0, 1) 0.05. Activations are f32 N(0, 1), a
feed-forward product's input N N'.

A case's fields:
  kind      "layer": a decoder layer's four products, launched one after
            another as an engine's step launches them: Q, K and V in one launch,
            the attention output, gate and up in one gated launch, down.
            "head": the LM head over the step's last token.
            "step": a whole decode step: the embedding gather, every layer, the
            head, captured once into a HIP graph and replayed, as a serving
            loop runs it.
            "encoder": an encoder's feed-forward pair: up with its bias and
            GELU, down with its bias, both clipped to four bounds.
  type      the weights' format;  head_type: a step's embedding and head
  tokens    rows of the step (1: decode)
  path      "auto" (the default), "split_f16" (the opt-in matrix-core
            prefill), "int8_limbs" (the opt-in decode)
Every step passes the engine's split gate and its range-sum buffer.
"""

import math

import torch

from charlotte_amd import matmul as mm

TYPES = {"f32": mm.TensorType.F32, "f16": mm.TensorType.F16, "q4_0": mm.TensorType.Q4_0, "q4_1": mm.TensorType.Q4_1,
         "q8_0": mm.TensorType.Q8_0, "q6_k": mm.TensorType.Q6_K, "bf16": mm.TensorType.BF16}
QUANTIZED = ("q4_0", "q4_1", "q8_0", "q6_k")
STORED = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q4_0": 18 / 32, "q4_1": 20 / 32, "q8_0": 34 / 32, "q6_k": 210 / 256}
CLIP = (-6.0, 6.0, -40.0, 40.0)

# The shapes of models this repository names: hidden, attention and
# feed-forward widths.
QWEN3_0_6B = {"hidden": 1024, "q": 2048, "kv": 1024, "ffn": 3072, "activation": "silu"}
LLAMA_3_2_1B = {"hidden": 2048, "q": 2048, "kv": 512, "ffn": 8192, "activation": "silu"}
LLAMA_3_8B = {"hidden": 4096, "q": 4096, "kv": 1024, "ffn": 14336, "activation": "silu"}
GEMMA_3_1B = {"hidden": 1152, "q": 1024, "kv": 256, "ffn": 6912, "activation": "gelu"}


def listed():
    layer = {"kind": "layer", "path": "auto"}
    return [
        # Decoding one token with a small model, the whole step: 28 layers of
        # small products, launch after launch, and the head.
        {"name": "decode_step", "kind": "step", "type": "q4_0", "head_type": "q6_k", "layers": 28, "vocab": 151936,
         "tokens": 1, "path": "auto", **QWEN3_0_6B},
        # The same model's layer launched call by call, as an engine that does
        # not capture its step runs it: the smallest work, the host's share with it.
        {"name": "decode_layer_small", **layer, "type": "q4_0", "tokens": 1, **QWEN3_0_6B},
        # Decoding with an 8B model: wide rows, bound by the weights' bytes.
        {"name": "decode_layer_wide", **layer, "type": "q4_0", "tokens": 1, **LLAMA_3_8B},
        # An unquantized file decoded as stored.
        {"name": "decode_layer_bf16", **layer, "type": "bf16", "tokens": 1, **LLAMA_3_2_1B},
        # LM heads, the largest single products of a decode step.
        {"name": "head_q6_k", "kind": "head", "type": "q6_k", "hidden": 1152, "vocab": 262144, "tokens": 1, "path": "auto"},
        {"name": "head_q8_0", "kind": "head", "type": "q8_0", "hidden": 2048, "vocab": 128256, "tokens": 1, "path": "auto"},
        # A few tokens at once: verifying drafted tokens, or a batch of sequences.
        {"name": "draft_5_tokens", **layer, "type": "q4_0", "tokens": 5, **LLAMA_3_2_1B},
        # A short chat turn over a cached prefix.
        {"name": "turn_21_tokens", **layer, "type": "q4_0", "tokens": 21, **LLAMA_3_2_1B},
        # A prompt of odd length, rows that straddle Q6_K super-blocks, GELU.
        {"name": "prompt_203_q6_k", **layer, "type": "q6_k", "tokens": 203, **GEMMA_3_1B},
        # The engine's prefill block, 512 tokens, on a small model.
        {"name": "prefill_512", **layer, "type": "q4_0", "tokens": 512, **QWEN3_0_6B},
        # A long prompt: compute-bound, the largest work.
        {"name": "prefill_2048", **layer, "type": "q4_0", "tokens": 2048, **LLAMA_3_2_1B},
        # The opt-in matrix-core prefill, which trades the fixed order of addition for speed.
        {"name": "prefill_512_split_f16", "kind": "layer", "type": "q4_0", "tokens": 512, "path": "split_f16", **LLAMA_3_2_1B},
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _wide(rng, low, high):
    """A width: most models' are multiples of 128 or more, some of 64 or 32 alone."""
    step = rng.choice([32, 64, 128, 256, 256, 512])
    return max(low, round(_log(rng, low, high) / step) * step)


def _tokens(rng):
    return 1 if rng.random() < 0.35 else int(round(_log(rng, 2, 2048)))


def _most(format_):
    """Weights times tokens, so that no step passes the longest prefill above."""
    return 40e9 if format_ == "f32" else 80e9


def draw(rng):
    """Another case of the ranges the listed ones stand for: widths of 512 to
    4,096 (feed-forward to four times that, at most 14,336) in whole 32s,
    vocabularies to 262,144 (odd ones among them), 1 to 2,048 tokens, every format."""
    pick = rng.random()
    kind = "head" if pick < 0.15 else "encoder" if pick < 0.3 else "layer"
    format_ = rng.choices(["q4_0", "q6_k", "q8_0", "q4_1", "bf16", "f16", "f32"], weights=[16, 7, 6, 4, 4, 4, 2])[0]
    if kind == "head":
        hidden = _wide(rng, 512, 4096)
        vocab = int(_log(rng, 16384, 262144))
        if format_ == "q6_k":
            vocab = vocab // 16 * 16
        vocab = min(vocab, int(280e6 / (hidden * STORED[format_])) // 16 * 16)
        limbs = format_ in ("q4_0", "q6_k") and rng.random() < 0.4
        return {"kind": kind, "type": format_, "hidden": hidden, "vocab": vocab,
                "tokens": 1 if limbs else _tokens(rng) % 64 + 1, "path": "int8_limbs" if limbs else "auto"}
    tokens = _tokens(rng)
    hidden = _wide(rng, 512, 4096)
    ffn = min(_wide(rng, 2 * hidden, 4 * hidden), 14336)
    if kind == "encoder":
        if rng.random() < 0.7:
            format_ = rng.choice(["f16", "bf16", "f32", "q8_0"])
        tokens = max(tokens, 16)
        weights = 2 * hidden * ffn
        tokens = max(2, min(tokens, int(_most(format_) / weights)))
        return {"kind": kind, "type": format_, "hidden": hidden, "ffn": ffn, "tokens": tokens, "path": "auto"}
    q = 64 * max(4, round(hidden * rng.choice([0.75, 1, 1, 2]) / 64))
    kv = 64 * max(1, q // (64 * rng.choice([1, 2, 4, 8])))
    weights = hidden * (q + 2 * kv) + q * hidden + 3 * hidden * ffn
    tokens = max(1, min(tokens, int(_most(format_) / weights)))
    split = format_ in QUANTIZED and tokens >= 16 and rng.random() < 0.15
    return {"kind": kind, "type": format_, "hidden": hidden, "q": q, "kv": kv, "ffn": ffn,
            "activation": rng.choice(["silu", "gelu"]), "tokens": tokens, "path": "split_f16" if split else "auto"}


# ---- a case's products: (key, epilogue, members' rows, K, activation) -----------


def _layer_products(c):
    return [("qkv", "qkv", [c["q"], c["kv"], c["kv"]], c["hidden"]), ("o", "write", [c["hidden"]], c["q"]),
            ("gate_up", "gated", [c["ffn"], c["ffn"]], c["hidden"]), ("down", "write", [c["hidden"]], c["ffn"])]


def _products(c):
    if c["kind"] == "layer":
        return [(p, c["type"]) for p in _layer_products(c)]
    if c["kind"] == "encoder":
        return [(("up", "encoder_up", [c["ffn"]], c["hidden"]), c["type"]),
                (("down", "encoder_down", [c["hidden"]], c["ffn"]), c["type"])]
    head = (("head", "last", [c["vocab"]], c["hidden"]), c.get("head_type", c["type"]))
    return [(p, c["type"]) for _ in range(c.get("layers", 0)) for p in _layer_products(c)] + [head]


# ---- weights in the device layout -------------------------------------------------


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _random_bytes(gen, n):
    return torch.randint(-(1 << 31), 1 << 31, ((n + 3) // 4,), generator=gen, device="cuda", dtype=torch.int64) \
        .to(torch.int32).view(torch.uint8)[:n]


def _scales(gen, n, size):
    return (_normal(gen, n).abs() * size).to(torch.float16)


def _piece(gen, format_, rows, columns):
    """A weight's piece in the device layout, a uint8 tensor."""
    n = rows * columns
    if format_ == "f32":
        return (_normal(gen, n) * 0.05).view(torch.uint8)
    if format_ in ("f16", "bf16"):
        return (_normal(gen, n) * 0.05).to(torch.float16 if format_ == "f16" else torch.bfloat16).view(torch.uint8)
    if format_ == "q6_k":
        blocks = n // 256
        scales = torch.randint(-64, 64, (16 * blocks,), generator=gen, device="cuda", dtype=torch.int8)
        parts = [_random_bytes(gen, 192 * blocks), scales.view(torch.uint8), _scales(gen, blocks, 0.001).view(torch.uint8)]
    else:
        blocks = n // 32
        codes = _random_bytes(gen, (32 if format_ == "q8_0" else 16) * blocks)
        d = _scales(gen, blocks, 0.0005 if format_ == "q8_0" else 0.02)
        if format_ == "q4_1":
            d = torch.stack([d, (d.float() * -8.0).to(torch.float16)], dim=1).reshape(-1)
        parts = [codes, d.view(torch.uint8)]
    out = torch.zeros(mm.layout_bytes(TYPES[format_], rows, columns), device="cuda", dtype=torch.uint8)
    at = 0
    for p in parts:
        out[at:at + p.numel()] = p
        at += p.numel()
    return out


def _weights64(piece, format_, rows, columns):
    """The piece's weights in 64 bits."""
    n = rows * columns
    if format_ in ("f32", "f16", "bf16"):
        kind = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[format_]
        return piece.view(kind).to(torch.float64).reshape(rows, columns)
    if format_ == "q6_k":
        b, g = n // 256, n // 32
        low = piece[:128 * b].reshape(g, 16)
        high = piece[128 * b:192 * b].reshape(g, 8)
        scales = piece[192 * b:208 * b].view(torch.int8).reshape(g, 2).to(torch.float64)
        d = piece[208 * b:210 * b].clone().view(torch.float16).to(torch.float64).repeat_interleave(8)
        q = torch.cat([low & 15, low >> 4], dim=1)
        pairs = torch.cat([(high >> (2 * i)) & 3 for i in range(4)], dim=1)
        w = (q | (pairs << 4)).to(torch.float64) - 32
        return (w.reshape(g, 2, 16) * (scales * d[:, None])[:, :, None]).reshape(rows, columns)
    g = n // 32
    if format_ == "q8_0":
        w = piece[:32 * g].view(torch.int8).to(torch.float64).reshape(g, 32)
        return (w * piece[32 * g:34 * g].clone().view(torch.float16).to(torch.float64)[:, None]).reshape(rows, columns)
    codes = piece[:16 * g].reshape(g, 16)
    w = torch.cat([codes & 15, codes >> 4], dim=1).to(torch.float64)
    if format_ == "q4_0":
        return ((w - 8) * piece[16 * g:18 * g].clone().view(torch.float16).to(torch.float64)[:, None]).reshape(rows, columns)
    dm = piece[16 * g:20 * g].clone().view(torch.float16).to(torch.float64).reshape(g, 2)
    return (w * dm[:, :1] + dm[:, 1:]).reshape(rows, columns)


# ---- inputs -------------------------------------------------------------------------


def _inputs(case, seed):
    """Everything a pass reads, from the seed alone: each product's pieces and
    input rows, an encoder's bounds and biases, a step's embedding table and token."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    tokens, products = case["tokens"], []
    for (key, epilogue, rows, columns), format_ in _products(case):
        p = {"key": key, "epilogue": epilogue, "rows": rows, "columns": columns, "type": format_,
             "pieces": [_piece(gen, format_, r, columns) for r in rows], "x": _normal(gen, tokens, columns)}
        if key == "down":
            p["x"] = p["x"] * _normal(gen, tokens, columns)
        if epilogue.startswith("encoder"):
            p["bias"] = _normal(gen, rows[0]) * 0.5
            p["clip"] = torch.tensor(CLIP, device="cuda", dtype=torch.float32)
        products.append(p)
    made = {"products": products}
    if case["kind"] == "step":
        made["ids"] = torch.randint(0, case["vocab"], (tokens,), generator=gen, device="cuda", dtype=torch.int32)
        made["table"] = _piece(gen, case["head_type"], case["vocab"], case["hidden"])
    return made


def _outputs(p, tokens):
    empty = lambda *shape: torch.zeros(*shape, device="cuda", dtype=torch.float32)  # noqa: E731
    if p["epilogue"] == "qkv":
        return [empty(tokens, r) for r in p["rows"]]
    return [empty(1 if p["epilogue"] == "last" else tokens, p["rows"][0])]


ACTIVATIONS = {"silu": mm.Activation.SiLU, "gelu": mm.Activation.GeluTanh}


def _launch_of(ctx, case, p, outputs):
    members = [mm.Member(mm.Weight(ctx, TYPES[p["type"]], r, p["columns"], device_piece=w.data_ptr(), nbytes=w.numel()))
               for r, w in zip(p["rows"], p["pieces"])]
    more = {"activation": ACTIVATIONS[case.get("activation", "gelu")]}
    if p["epilogue"] == "qkv":
        more["epilogue"] = mm.Epilogue.QKV
    elif p["epilogue"] == "gated":
        more["epilogue"] = mm.Epilogue.GatedActivation
    elif p["epilogue"] == "last":
        more["rows"] = mm.Rows.LastToken
    elif p["epilogue"].startswith("encoder"):
        more["bias"], more["activated"] = p["bias"].data_ptr(), p["epilogue"] == "encoder_up"
        more["clip"] = [p["clip"].data_ptr() + 4 * i for i in range(4)]
    return mm.MatmulLaunch(members, p["x"].data_ptr(), [o.data_ptr() for o in outputs], **more)


def prepare(case, seed):
    s = _inputs(case, seed)
    tokens = case["tokens"]
    ctx = mm.Context(torch.cuda.current_device())
    s["ctx"], s["tokens"] = ctx, tokens
    s["stream"] = torch.cuda.current_stream().cuda_stream
    if case["kind"] == "step":  # a buffer a product, every layer's outputs in it
        count, head = case["layers"], s["products"][-1]
        s["by_product"] = [[torch.stack([t] * count) for t in _outputs(p, tokens)] for p in s["products"][:4]]
        s["outputs"] = [[t[i // 4] for t in s["by_product"][i % 4]] for i in range(4 * count)] + [_outputs(head, tokens)]
    else:
        s["outputs"] = [_outputs(p, tokens) for p in s["products"]]
    s["launches"] = [_launch_of(ctx, case, p, o) for p, o in zip(s["products"], s["outputs"])]
    # the engine's range sums: what its gate lets the largest split take
    floats = 0
    for p, m in zip(s["products"], s["launches"]):
        if m.rows == mm.Rows.EveryToken and tokens > 1:
            floats = max(floats, mm.range_sum_floats(m.epilogue, sum(p["rows"]), p["columns"], mm.kSplitGate))
    s["sums"] = torch.zeros(max(floats, 4), device="cuda", dtype=torch.float32)
    s["sums_at"], s["sums_bytes"] = (s["sums"].data_ptr(), 4 * floats) if floats else (0, 0)
    if case["path"] == "split_f16":
        nbytes = max(mm.workspace_bytes(tokens, p["columns"]) for p in s["products"])
        s["workspace"] = torch.empty(nbytes, device="cuda", dtype=torch.uint8)
        ctx.set_gemm_path(mm.GemmPath.SPLIT_F16_MFMA)
        ctx.set_workspace(s["workspace"].data_ptr(), nbytes)
    elif case["path"] == "int8_limbs":
        ctx.set_gemv_path(mm.GemvPath.INT8_LIMBS)
    if case["kind"] == "step":
        s["hidden"] = torch.zeros(tokens, case["hidden"], device="cuda", dtype=torch.float32)
        s["embedding"] = mm.Weight(ctx, TYPES[case["head_type"]], case["vocab"], case["hidden"],
                                   device_piece=s["table"].data_ptr(), nbytes=s["table"].numel())
        _step(s, s["stream"])  # the first pass, before the capture
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s, torch.cuda.current_stream().cuda_stream)
    return s


def _step(s, stream):
    ctx, tokens = s["ctx"], s["tokens"]
    mm.gather(ctx, s["embedding"], s["ids"].data_ptr(), tokens, s["hidden"].data_ptr(), stream=stream)
    for m in s["launches"]:
        mm.launch(ctx, m, tokens, stream=stream)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return [state["hidden"], state["by_product"], state["outputs"][-1]]
    ctx, tokens, stream = state["ctx"], state["tokens"], state["stream"]
    at, nbytes = state["sums_at"], state["sums_bytes"]
    for m in state["launches"]:
        mm.launch(ctx, m, tokens, mm.kSplitGate, at, nbytes, stream)
    return state["outputs"]


# ---- what a pass cannot do without -----------------------------------------------------


def work(case):
    tokens, nbytes, flops = case["tokens"], 0.0, 0.0
    for (_, epilogue, rows, columns), format_ in _products(case):
        t = 1 if epilogue == "last" else tokens
        weights = sum(rows) * columns
        written = rows[0] if epilogue == "gated" else sum(rows)
        nbytes += weights * STORED[format_] + 4 * t * (columns + written)
        flops += 2 * t * weights
    if case["kind"] == "step":
        nbytes += tokens * case["hidden"] * (4 + STORED[case["head_type"]])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Every default path adds in one documented order, so a correct kernel
    # gives the same bits. The two opt-in paths keep about 22 bits of each
    # input: the split-f16 prefill measures 3e-7 from 64 bits (2-norm), the
    # int8-limb decode as much.
    if case["path"] in ("split_f16", "int8_limbs"):
        return {"rel": 2e-6, "max": 2e-5}
    return "exact"


def _activate64(name, g):
    if name == "silu":
        return g * torch.sigmoid(g)
    return 0.5 * g * (1 + torch.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))


def exact(case, seed):
    """A pass's outputs in 64 bits, by plain torch."""
    made, activation, outputs = _inputs(case, seed), case.get("activation", "gelu"), []
    for p in made["products"]:
        x = p["x"].to(torch.float64)
        if p["epilogue"] == "last":
            x = x[-1:]
        if "clip" in p:
            x = x.clamp(CLIP[0], CLIP[1])
        y = [x @ _weights64(w, p["type"], r, p["columns"]).t() for w, r in zip(p["pieces"], p["rows"])]
        if p["epilogue"] == "gated":
            y = [_activate64(activation, y[0]) * y[1]]
        if "clip" in p:
            y = [y[0].clamp(CLIP[2], CLIP[3]) + p["bias"].to(torch.float64)]
            if p["epilogue"] == "encoder_up":
                y = [_activate64("gelu", y[0])]
        outputs.append(y)
        p["pieces"] = None
    if case["kind"] == "step":
        table = made["table"]
        rows = _weights64(table, case["head_type"], case["vocab"], case["hidden"])[made["ids"].long()]
        by_product = [[torch.stack(t) for t in zip(*outputs[i:-1:4])] for i in range(4)]
        return [rows, by_product, outputs[-1]]
    return outputs
