"""What a user of this framework runs, as cases that can be timed and checked.

Five kinds of work, each through the public entry points:

* ``linear``: one ``PackedW3Linear`` called eagerly, any shape, one to eight rows
  on the packed route, more on the dense fallback.
* ``step``: the Linears of one decode token, bound and captured in one graph as a
  serving loop keeps them: the seven Linears of a Qwen3-8B decoder layer for
  several layers (W3 or hybrid two-base), or the rank-one two-base gate GEMVs.
* ``prefill``: the seven Linears of a layer on many rows, called eagerly as the
  model's prefill calls them (``fallback="dense"``).
* ``norm_rope``: the fused RMSNorm, q/k norm and RoPE of a layer on a sequence.
* ``decode``: a ``NativeDecodeSession`` over a few full-size layers and the full
  vocabulary: a replay of its captured continuation, returning the logits.

Weights are drawn as quantized checkpoints have them: bell-shaped 3-bit codes
around the zero-point, scales U[0.005, 0.02], and either the identity column
order or the desc_act order of a GPTQ checkpoint.
"""
from __future__ import annotations

import math

import torch

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM, VOCAB = 4096, 12288, 32, 8, 128, 151936
EPS, THETA = 1e-6, 1_000_000.0
# name: (out_features, in_features, the input it reads)
LAYER = {
    "self_attn.q_proj": (4096, 4096, "hidden"), "self_attn.k_proj": (1024, 4096, "hidden"),
    "self_attn.v_proj": (1024, 4096, "hidden"), "self_attn.o_proj": (4096, 4096, "attn"),
    "mlp.gate_proj": (12288, 4096, "hidden2"), "mlp.up_proj": (12288, 4096, "hidden2"),
    "mlp.down_proj": (4096, 12288, "act"),
}
INPUT_WIDTH = {"hidden": 4096, "attn": 4096, "hidden2": 4096, "act": 12288}


def listed():
    return [
        # the smallest call: one row through a small odd Linear with a bias, eagerly;
        # call latency and launches are what it costs
        {"name": "linear_odd_1", "kind": "linear", "out": 1000, "in": 1408, "rows": 1, "packed_rows": 1,
         "dtype": "bf16", "scale": "bf16", "zeros": True, "order": "desc_act", "bias": True},
        # a decode token's Linears, the benchmark's own step: 8 layers, fp16 scales, zero-points
        {"name": "step_w3", "kind": "step", "format": "w3", "layers": 8, "rows": 1, "route": "structural",
         "dtype": "bf16", "scale": "f16", "zeros": True, "order": "identity"},
        # the same token on a real GPTQ checkpoint (desc_act, bf16 scales, zero 4) with the
        # reference's observed_exact route
        {"name": "step_w3_exact", "kind": "step", "format": "w3", "layers": 2, "rows": 1, "route": "observed_exact",
         "dtype": "bf16", "scale": "bf16", "zeros": False, "order": "desc_act"},
        # eight sequences decoded together on the packed route
        {"name": "step_w3_rows8", "kind": "step", "format": "w3", "layers": 2, "rows": 8, "route": "structural",
         "dtype": "bf16", "scale": "f16", "zeros": True, "order": "identity"},
        # a decode token on the hybrid two-base format
        {"name": "step_hybrid", "kind": "step", "format": "hybrid", "layers": 2, "rows": 1, "dtype": "bf16"},
        # the rank-one two-base gate GEMV (12288 x 4096, 32 salient columns) of four layers
        {"name": "step_rank_one", "kind": "step", "format": "rank_one", "layers": 4, "out": 12288, "in": 4096,
         "salient": 32, "rows": 1, "dtype": "bf16"},
        # a short prompt, or a batch of more sequences than the packed route takes
        {"name": "prefill_w3_37", "kind": "prefill", "format": "w3", "rows": 37, "dtype": "bf16", "scale": "bf16",
         "zeros": False, "order": "desc_act"},
        # the benchmark's 512-token prompt
        {"name": "prefill_w3_512", "kind": "prefill", "format": "w3", "rows": 512, "dtype": "bf16", "scale": "bf16",
         "zeros": False, "order": "desc_act"},
        # the largest: a 2048-token chunk in fp16
        {"name": "prefill_w3_2048", "kind": "prefill", "format": "w3", "rows": 2048, "dtype": "f16", "scale": "f16",
         "zeros": True, "order": "identity"},
        # a prompt on the hybrid two-base format
        {"name": "prefill_hybrid_200", "kind": "prefill", "format": "hybrid", "rows": 200, "dtype": "bf16"},
        # the fused modules of one layer over a prompt
        {"name": "norm_rope_1000", "kind": "norm_rope", "tokens": 1000, "dtype": "bf16"},
        # whole decode: 4 layers, 512 tokens of context, 8 tokens, LM head
        {"name": "decode_w3", "kind": "decode", "layers": 4, "prefix": 512, "steps": 8, "zeros": True,
         "scale": "f16", "order": "identity"},
    ]


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    half = rng.choice(("bf16", "bf16", "f16"))
    w3 = {"scale": rng.choice(("bf16", "f16")), "zeros": rng.random() < 0.5,
          "order": rng.choice(("identity", "desc_act"))}
    kind = rng.choice(("linear", "linear", "step", "step", "prefill", "prefill", "norm_rope", "decode"))
    if kind == "linear":
        rows = log_int(1, 2048)
        return {"kind": kind, "out": log_int(16, 16384), "in": 128 * log_int(1, 96), "rows": rows,
                "packed_rows": 8 if rng.random() < 0.5 else 1, "dtype": half, "bias": rng.random() < 0.3, **w3}
    if kind == "step":
        fmt = rng.choice(("w3", "w3", "w3", "hybrid", "rank_one"))
        base = {"kind": kind, "format": fmt, "layers": rng.randint(1, 4), "rows": 1, "dtype": half}
        if fmt == "hybrid":
            return base
        if fmt == "rank_one":
            return {**base, "out": log_int(1024, 16384), "in": 128 * rng.randint(16, 96),
                    "salient": rng.randint(0, 32)}
        route = rng.choice(("structural", "structural", "fast_corrected", "observed_exact"))
        if route != "structural":
            w3["scale"] = "bf16"  # these routes take bf16 scales
        return {**base, "rows": rng.randint(1, 8) if route == "structural" else 1, "route": route, **w3}
    if kind == "prefill":
        fmt = rng.choice(("w3", "w3", "w3", "hybrid"))
        if fmt == "hybrid":
            return {"kind": kind, "format": fmt, "rows": log_int(2, 1024), "dtype": half}
        return {"kind": kind, "format": fmt, "rows": log_int(9, 1536), "dtype": half, **w3}
    if kind == "norm_rope":
        return {"kind": kind, "tokens": log_int(1, 4096), "dtype": half}
    return {"kind": kind, "layers": rng.randint(1, 4), "prefix": log_int(16, 1024), "steps": rng.randint(1, 8), **w3}


# ------------------------------------------------------------------ inputs
def _generators(seed):
    return (torch.Generator(device=DEVICE).manual_seed(seed), torch.Generator().manual_seed(seed))


def _desc_act(k, cpu):
    """A GPTQ desc_act column order: each group of 128 holds a random ascending
    subset of the columns."""
    order = torch.randperm(k, generator=cpu)
    group = torch.empty(k, dtype=torch.int64)
    group[order] = torch.arange(k) // 128
    return torch.argsort(group, stable=True).to(torch.int16).to(DEVICE)


def _w3_draw(o, k, gen, scale, zeros, perm):
    """Codes in sorted column order uint8 [G, 128, O], scales [G, O], zero-points or None, perm."""
    g = k // 128
    spread = torch.randn((g, 128, o), generator=gen, device=DEVICE, dtype=torch.float16)
    zero = (torch.randint(3, 5, (g, o), generator=gen, device=DEVICE, dtype=torch.uint8) if zeros else None)
    codes = (spread * 1.6 + 4.0).round_().clamp_(0, 7).to(torch.uint8)
    scales = (torch.rand((g, o), generator=gen, device=DEVICE) * 0.015 + 0.005).to(DTYPES[scale])
    return codes, scales, zero, perm


def _w3_layout(drawn):
    """The planar payload of drawn codes: bit p of the code of column 8c + j of a
    group is bit j of byte c of plane p, plane 2 inverted."""
    codes, scales, zero, perm = drawn
    g, _, o = codes.shape
    columns = codes.reshape(g, 16, 8, o)
    planes = torch.empty((g, 3, o, 16), dtype=torch.uint8, device=DEVICE)
    for p in range(3):
        byte = torch.zeros((g, 16, o), dtype=torch.uint8, device=DEVICE)
        for j in range(8):
            byte |= ((columns[:, :, j] >> p) & 1) << j
        planes[:, p] = (byte if p < 2 else ~byte).permute(0, 2, 1)
    layout = {"planes": planes, "scales": scales, "perm": perm}
    if zero is not None:
        layout["zeros"] = zero
    return layout


def _identity(k):
    return torch.arange(k, dtype=torch.int16, device=DEVICE)


def _layer_perms(order, cpu):
    """One column order per layer input: Linears that read the same input share it."""
    return {name: _desc_act(width, cpu) if order == "desc_act" else _identity(width)
            for name, width in INPUT_WIDTH.items()}


def _w3_layer(case, gen, cpu):
    perms = _layer_perms(case["order"], cpu)
    return {name: _w3_draw(o, k, gen, case["scale"], case["zeros"], perms[src])
            for name, (o, k, src) in LAYER.items()}


def _hybrid_draw(o, k, gen):
    """The seven payload fields: two {-1, +1} bases, two bits a column and four
    columns a byte, per-group row and column scales, and eight refined columns a
    group.  Scales are those of trained factors: row scales of the weight's size,
    column scales around one."""
    g = k // 128

    def scale(shape, mean, spread):
        return mean * (1 + spread * torch.randn(shape, generator=gen, device=DEVICE))

    refined = torch.rand((g, 128), generator=gen, device=DEVICE).argsort(dim=1)[:, :8].sort(dim=1).values
    base = torch.tensor([1.0, 0.5], device=DEVICE)
    return {
        "global_sign_codes": torch.randint(0, 256, (o, 32 * g), generator=gen, device=DEVICE, dtype=torch.uint8),
        "global_row_scales": base[:, None, None] * scale((2, o, g), 0.015, 0.2),
        "global_column_scales": scale((2, g, 128), 1.0, 0.2),
        "refinement_indices": refined.to(torch.int16),
        "refinement_sign_codes": torch.randint(0, 256, (o, 2 * g), generator=gen, device=DEVICE, dtype=torch.uint8),
        "refinement_row_scales": 0.5 * base[:, None, None] * scale((2, o, g), 0.015, 0.2),
        "refinement_column_scales": scale((2, g, 8), 1.0, 0.2),
    }


def _rank_one_draw(o, k, s, gen):
    layout = {
        "planes": torch.randint(0, 256, (k // 128, o, 2, 16), generator=gen, device=DEVICE, dtype=torch.uint8),
        "coef": (0.3 + 0.5 * torch.rand((2, o), generator=gen, device=DEVICE)).half(),
        "srow": (0.01 + 0.02 * torch.rand(o, generator=gen, device=DEVICE)).half(),
        "tcol": (0.5 + torch.rand(k, generator=gen, device=DEVICE)).half(),
    }
    if s:
        layout["salient"] = (0.05 * torch.randn((o, s), generator=gen, device=DEVICE)).to(torch.bfloat16)
        layout["salient_idx"] = torch.rand(k, generator=gen, device=DEVICE).argsort()[:s].sort().values.int()
    return layout


def _activations(rows, width, dtype, gen, source="hidden"):
    """Normalised hidden states with a few strong channels, or SwiGLU outputs."""
    x = torch.randn((rows, width), generator=gen, device=DEVICE)
    if source == "act":
        x = x * torch.nn.functional.silu(torch.randn((rows, width), generator=gen, device=DEVICE))
    elif width >= 1024:
        x[:, torch.randint(0, width, (4,), generator=gen, device=DEVICE)] *= 20.0
    return x.to(DTYPES[dtype])


def _layer_inputs(rows, dtype, gen):
    return {name: _activations(rows, width, dtype, gen, name) for name, width in INPUT_WIDTH.items()}


def _rows_shape(rows, width):
    return (1, rows, width)


# ------------------------------------------------------------------ prepare
def _capture(fn):
    """``fn`` captured as a serving loop does: warmed up on a side stream, then recorded."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        outputs = fn()
    return graph, outputs


def _w3_module(drawn, **kwargs):
    from marlin_style_fluxbin_amd import PackedW3Linear

    return PackedW3Linear(_w3_layout(drawn), **kwargs)


def _draw_linear(case, seed):
    gen, cpu = _generators(seed)
    o, k = case["out"], case["in"]
    perm = _desc_act(k, cpu) if case["order"] == "desc_act" else _identity(k)
    drawn = _w3_draw(o, k, gen, case["scale"], case["zeros"], perm)
    bias = (0.1 * torch.randn(o, generator=gen, device=DEVICE)).to(DTYPES[case["dtype"]]) if case["bias"] else None
    return drawn, bias, _activations(case["rows"], k, case["dtype"], gen)


def _prepare_linear(case, seed):
    drawn, bias, x = _draw_linear(case, seed)
    module = _w3_module(drawn, bias=bias, fallback="dense", row_tile=256, max_packed_rows=case["packed_rows"])
    return {"kind": "linear", "module": module.eval(), "x": x}


def _prepare_step(case, seed):
    gen, cpu = _generators(seed)
    dtype = DTYPES[case["dtype"]]
    calls = []
    if case["format"] == "rank_one":
        from marlin_style_fluxbin_amd import TwoBaseGemv

        for _ in range(case["layers"]):
            gemv = TwoBaseGemv(_rank_one_draw(case["out"], case["in"], case["salient"], gen))
            x = _activations(1, case["in"], case["dtype"], gen)
            out = torch.empty((1, case["out"]), dtype=dtype, device=DEVICE)
            calls.append((gemv, (x, out)))
    else:
        for _ in range(case["layers"]):
            if case["format"] == "w3":
                from marlin_style_fluxbin_amd import qwen3_w3_route

                modules = {}
                for name, drawn in _w3_layer(case, gen, cpu).items():
                    o, k, _ = LAYER[name]
                    modules[name] = _w3_module(drawn, route=case["route"], max_packed_rows=max(case["rows"], 1),
                                               **qwen3_w3_route(case["route"], o, k))
            else:
                from marlin_style_fluxbin_amd import PackedHybridLinear

                modules = {name: PackedHybridLinear(_hybrid_draw(o, k, gen), kernel="v5_p1024")
                           for name, (o, k, _) in LAYER.items()}
            inputs = _layer_inputs(case["rows"], case["dtype"], gen)
            for name, module in modules.items():
                _, k, src = LAYER[name]
                if case["rows"] == 1:
                    module.bind_prepared_decode(dtype)
                calls.append((module, (inputs[src].view(_rows_shape(case["rows"], k)),)))
    with torch.inference_mode():
        graph, outputs = _capture(lambda: [fn(*args) for fn, args in calls])
    return {"kind": "step", "graph": graph, "outputs": outputs, "keep": calls}


def _prepare_prefill(case, seed):
    gen, cpu = _generators(seed)
    if case["format"] == "w3":
        modules = {name: _w3_module(drawn, fallback="dense") for name, drawn in _w3_layer(case, gen, cpu).items()}
    else:
        from marlin_style_fluxbin_amd import PackedHybridLinear

        modules = {name: PackedHybridLinear(_hybrid_draw(o, k, gen), kernel="v5_p1024", fallback="dense")
                   for name, (o, k, _) in LAYER.items()}
    inputs = _layer_inputs(case["rows"], case["dtype"], gen)
    calls = [(module, inputs[LAYER[name][2]].view(_rows_shape(case["rows"], LAYER[name][1])))
             for name, module in modules.items()]
    return {"kind": "prefill", "calls": calls}


def _rope_tables(positions, dtype):
    inv = THETA ** (-torch.arange(0, HEAD_DIM, 2, dtype=torch.float64) / HEAD_DIM)
    angles = torch.cat([positions.double()[:, None] * inv] * 2, dim=1)
    return angles.cos().to(DEVICE, dtype)[None], angles.sin().to(DEVICE, dtype)[None]


def _draw_norm_rope(case, seed):
    gen, _ = _generators(seed)
    t, dtype = case["tokens"], DTYPES[case["dtype"]]

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=DEVICE).to(dtype)

    def weight(n):
        return (1 + 0.1 * torch.randn(n, generator=gen, device=DEVICE)).to(dtype)

    cos, sin = _rope_tables(torch.arange(t), dtype)
    return {"hidden": _activations(t, HIDDEN, case["dtype"], gen)[None], "q": normal(1, t, HEADS, HEAD_DIM),
            "k": normal(1, t, KV_HEADS, HEAD_DIM), "hidden_weight": weight(HIDDEN), "q_weight": weight(HEAD_DIM),
            "k_weight": weight(HEAD_DIM), "cos": cos, "sin": sin}


def _draw_decode(case, seed):
    """Every weight of a small-depth Qwen3-8B: W3 layers, norms, embedding, head; and the tokens."""
    gen, cpu = _generators(seed)

    def dense(rows, std):
        return (std * torch.randn((rows, HIDDEN), generator=gen, device=DEVICE)).to(torch.bfloat16)

    def norm(n):
        return (1 + 0.1 * torch.randn(n, generator=gen, device=DEVICE)).to(torch.bfloat16)

    weights = {"embed": dense(VOCAB, 1.0), "head": dense(VOCAB, 0.02), "norm": norm(HIDDEN), "layers": []}
    for _ in range(case["layers"]):
        weights["layers"].append({"linears": _w3_layer(case, gen, cpu), "in": norm(HIDDEN), "post": norm(HIDDEN),
                                  "q": norm(HEAD_DIM), "k": norm(HEAD_DIM)})
    tokens = torch.randint(0, VOCAB, (1, case["prefix"] + case["steps"]), generator=cpu).to(DEVICE)
    return weights, tokens


def _prepare_decode(case, seed):
    from marlin_style_fluxbin_amd import replace_w3_block_linears
    from marlin_style_fluxbin_amd.native_decode import NativeDecodeSession
    from marlin_style_fluxbin_amd.qwen3 import qwen3_config, random_qwen3_model

    weights, tokens = _draw_decode(case, seed)
    model = random_qwen3_model(qwen3_config(num_hidden_layers=case["layers"]), device=DEVICE, dtype=torch.bfloat16)
    with torch.no_grad():
        model.model.embed_tokens.weight.copy_(weights["embed"])
        model.lm_head.weight.copy_(weights["head"])
        model.model.norm.weight.copy_(weights["norm"])
        for block, layer in zip(model.model.layers, weights["layers"]):
            block.input_layernorm.weight.copy_(layer["in"])
            block.post_attention_layernorm.weight.copy_(layer["post"])
            block.self_attn.q_norm.weight.copy_(layer["q"])
            block.self_attn.k_norm.weight.copy_(layer["k"])
            payload = {f"{name}.{field}": value for name, drawn in layer["linears"].items()
                       for field, value in _w3_layout(drawn).items()}
            replace_w3_block_linears(block, payload, fallback="dense")
    session = NativeDecodeSession(model, tokens[:, :case["prefix"]], tokens[:, case["prefix"]:])
    session.capture()
    return {"kind": "decode", "session": session}


def prepare(case, seed):
    if case["kind"] == "norm_rope":
        return {"kind": "norm_rope", **_draw_norm_rope(case, seed)}
    with torch.no_grad():
        return {"linear": _prepare_linear, "step": _prepare_step, "prefill": _prepare_prefill,
                "decode": _prepare_decode}[case["kind"]](case, seed)


# ------------------------------------------------------------------ run
def run(state):
    kind = state["kind"]
    if kind == "step":
        state["graph"].replay()
        return state["outputs"]
    if kind == "decode":
        state["session"].graph.replay()
        return state["session"].logits
    with torch.inference_mode():
        if kind == "linear":
            return state["module"](state["x"])
        if kind == "prefill":
            return [module(x) for module, x in state["calls"]]
        from marlin_style_fluxbin_amd import fused_apply_rotary_pos_emb, rms_norm

        hidden = rms_norm(state["hidden"], state["hidden_weight"], EPS)
        q = rms_norm(state["q"], state["q_weight"], EPS).transpose(1, 2)
        k = rms_norm(state["k"], state["k_weight"], EPS).transpose(1, 2)
        return [hidden, *fused_apply_rotary_pos_emb(q, k, state["cos"], state["sin"])]


# ------------------------------------------------------------------ work
def _linear_work(fmt, o, k, rows, case):
    g = k // 128
    io = 2 * rows * (k + o)
    if fmt == "w3":
        payload = 3 * o * k // 8 + 2 * g * o + (g * o if case["zeros"] else 0)
        payload += 2 * k if case["order"] == "desc_act" else 0
    elif fmt == "hybrid":  # signs, row scales, column scales, refinement
        payload = o * k // 4 + 8 * g * o + 8 * k + 16 * g + 2 * g * o + 8 * g * o + 64 * g
    else:
        s = case["salient"]
        payload = o * k // 4 + 6 * o + 2 * k + 2 * s * o + 4 * s
    return payload + io, 2 * rows * o * k


def work(case):
    kind = case["kind"]
    if kind == "linear":
        total, flops = _linear_work("w3", case["out"], case["in"], case["rows"], case)
        return {"bytes": total, "flops": flops}
    if kind in ("step", "prefill"):
        shapes = ([(case["out"], case["in"])] if case["format"] == "rank_one"
                  else [(o, k) for o, k, _ in LAYER.values()])
        per = [_linear_work(case["format"], o, k, case["rows"], case) for o, k in shapes]
        layers = case.get("layers", 1)
        return {"bytes": layers * sum(b for b, _ in per), "flops": layers * sum(f for _, f in per)}
    if kind == "norm_rope":
        t = case["tokens"]
        heads = (HEADS + KV_HEADS) * HEAD_DIM
        return {"bytes": 4 * t * (HIDDEN + heads) + 4 * t * HEAD_DIM + 2 * (HIDDEN + 2 * HEAD_DIM),
                "flops": 4 * t * HIDDEN + 10 * t * heads}
    per = [_linear_work("w3", o, k, 1, {**case, "order": "identity"}) for o, k, _ in LAYER.values()]
    total = flops = 0
    for i in range(case["steps"]):
        keys = case["prefix"] + i + 1
        total += case["layers"] * (sum(b for b, _ in per) + 4 * KV_HEADS * HEAD_DIM * keys)
        flops += case["layers"] * (sum(f for _, f in per) + 4 * HEADS * HEAD_DIM * keys)
        total += 2 * VOCAB * HIDDEN + 2 * VOCAB
        flops += 2 * VOCAB * HIDDEN
    return {"bytes": total, "flops": flops}


# ------------------------------------------------------------------ tolerance
def tolerance(case):
    """Outputs are rounded once to bf16 (2^-9 relative at most, 1.7e-3 in the mean)
    or fp16 (an eighth of that) from 32-bit sums; the dense fallback also rounds
    each weight.  A whole decode carries the roundings of every layer."""
    if case["kind"] == "decode":
        return {"rel": 1.6e-2, "max": 0.1}
    if case["dtype"] == "f16":
        return {"rel": 1.5e-3, "max": 1e-2}
    return {"rel": 7e-3, "max": 4e-2}


# ------------------------------------------------------------------ exact
def _w3_weight(drawn, rounding=()):
    """[O, K] in 64 bits, original column order; ``rounding``: the types that each
    weight is rounded to in turn (the dense fallback, the decoded_bf16 routes)."""
    codes, scales, zero, perm = drawn
    g, _, o = codes.shape
    z = zero.double() if zero is not None else torch.full((g, o), 4.0, dtype=torch.float64, device=DEVICE)
    w = (codes.double() - z[:, None]) * scales.double()[:, None]
    for dtype in rounding:
        w = w.float().to(dtype).double()  # the product of a half scale and a small integer fits 32 bits
    w = w.reshape(g * 128, o)
    dense = torch.empty_like(w)
    dense[perm.long()] = w
    return dense.t()


def _signs(codes, columns):
    """Two bases [2, O, K] from four columns a byte, base b of column i at bit 2 i + b."""
    bits = (codes[:, :, None].int() >> torch.arange(8, device=DEVICE, dtype=torch.int32)) & 1
    bits = bits.reshape(codes.shape[0], -1, 2)[:, :columns]
    return (bits.double() * 2 - 1).permute(2, 0, 1)


def _hybrid_weight(p, dtype=None):
    o, g = p["global_row_scales"].shape[1:]
    w = torch.zeros((o, g, 128), dtype=torch.float64, device=DEVICE)
    signs = _signs(p["global_sign_codes"], 128 * g).reshape(2, o, g, 128)
    extra = torch.zeros((o, g, 8), dtype=torch.float64, device=DEVICE)
    refined = _signs(p["refinement_sign_codes"], 8 * g).reshape(2, o, g, 8)
    for b in range(2):
        w += signs[b] * p["global_row_scales"][b].double()[:, :, None] * p["global_column_scales"][b].double()
        extra += (refined[b] * p["refinement_row_scales"][b].double()[:, :, None]
                  * p["refinement_column_scales"][b].double())
    w.scatter_add_(2, p["refinement_indices"].long()[None].expand(o, -1, -1), extra)
    w = w.reshape(o, g * 128)
    return w if dtype is None else w.float().to(dtype).double()


def _rank_one_weight(p):
    g, o = p["planes"].shape[:2]
    bits = (p["planes"][:, :, :, None, :].int() >> torch.arange(8, device=DEVICE, dtype=torch.int32)[:, None]) & 1
    signs = bits.reshape(g, o, 2, 128).permute(2, 1, 0, 3).reshape(2, o, g * 128).double() * 2 - 1
    coef = p["coef"].double()
    w = p["srow"].double()[:, None] * p["tcol"].double() * (coef[0][:, None] * signs[0] + coef[1][:, None] * signs[1])
    if "salient" in p:
        w.index_add_(1, p["salient_idx"].long(), p["salient"].double())
    return w


def _exact_linear(case, seed):
    drawn, bias, x = _draw_linear(case, seed)
    dense = case["rows"] > case["packed_rows"]
    w = _w3_weight(drawn, (DTYPES[case["scale"]], DTYPES[case["dtype"]]) if dense else ())
    y = x.double() @ w.t()
    return y if bias is None else y + bias.double()


def _exact_layers(case, seed):
    gen, cpu = _generators(seed)
    dtype, rows, found = DTYPES[case["dtype"]], case["rows"], []
    if case["format"] == "rank_one":
        for _ in range(case["layers"]):
            w = _rank_one_weight(_rank_one_draw(case["out"], case["in"], case["salient"], gen))
            found.append(_activations(1, case["in"], case["dtype"], gen).double() @ w.t())
        return found
    for _ in range(case.get("layers", 1)):
        if case["format"] == "w3":
            drawn = _w3_layer(case, gen, cpu)
        else:
            drawn = {name: _hybrid_draw(o, k, gen) for name, (o, k, _) in LAYER.items()}
        inputs = _layer_inputs(rows, case["dtype"], gen)
        for name, (o, k, src) in LAYER.items():
            dense = case["kind"] == "prefill"
            if case["format"] == "hybrid":
                w = _hybrid_weight(drawn[name], dtype if dense else None)
            elif dense:
                w = _w3_weight(drawn[name], (DTYPES[case["scale"]], dtype))
            else:
                w = _w3_weight(drawn[name], () if case["route"] == "structural" else (torch.bfloat16,))
            found.append((inputs[src].double() @ w.t()).view(_rows_shape(rows, o)))
    return found


def _norm64(x, weight):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin


def _exact_norm_rope(case, seed):
    s = _draw_norm_rope(case, seed)
    cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]
    q = _norm64(s["q"].double(), s["q_weight"]).transpose(1, 2)
    k = _norm64(s["k"].double(), s["k_weight"]).transpose(1, 2)
    return [_norm64(s["hidden"].double(), s["hidden_weight"]), _rope64(q, cos, sin), _rope64(k, cos, sin)]


def _exact_decode(case, seed):
    """The whole sequence at once, causally, in 64 bits: logits of the continuation's tokens."""
    weights, tokens = _draw_decode(case, seed)
    t = tokens.shape[1]
    cos, sin = _rope_tables(torch.arange(t), torch.float64)
    mask = torch.ones((t, t), dtype=torch.bool, device=DEVICE).triu(1)
    h = weights["embed"][tokens[0]].double()
    for layer in weights["layers"]:
        def linear(name, x):
            return x @ _w3_weight(layer["linears"][name]).t()

        x = _norm64(h, layer["in"])
        q = _norm64(linear("self_attn.q_proj", x).view(t, HEADS, HEAD_DIM), layer["q"]).transpose(0, 1)
        k = _norm64(linear("self_attn.k_proj", x).view(t, KV_HEADS, HEAD_DIM), layer["k"]).transpose(0, 1)
        v = linear("self_attn.v_proj", x).view(t, KV_HEADS, HEAD_DIM).transpose(0, 1)
        q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
        k, v = (a.repeat_interleave(HEADS // KV_HEADS, dim=0) for a in (k, v))
        scores = (q @ k.transpose(1, 2)) / math.sqrt(HEAD_DIM)
        attn = scores.masked_fill(mask, float("-inf")).softmax(-1) @ v
        h = h + linear("self_attn.o_proj", attn.transpose(0, 1).reshape(t, HEADS * HEAD_DIM))
        x = _norm64(h, layer["post"])
        gate = torch.nn.functional.silu(linear("mlp.gate_proj", x))
        h = h + linear("mlp.down_proj", gate * linear("mlp.up_proj", x))
    last = _norm64(h[case["prefix"]:], weights["norm"])
    return torch.cat([last @ part.double().t() for part in weights["head"].split(16384)], dim=1)


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "linear":
            return _exact_linear(case, seed)
        if case["kind"] in ("step", "prefill"):
            return _exact_layers(case, seed)
        if case["kind"] == "norm_rope":
            return _exact_norm_rope(case, seed)
        return _exact_decode(case, seed)
