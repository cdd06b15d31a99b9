"""The framework's work, as a program that serves a model with it calls it.

Each case goes through a public entry point (a facade under `kernels`, or the decode
attention call of `runtime.ops`). A decode step is run as programs run it here: the
calls of a few layers captured once in a graph and replayed, each layer with weights or a
cache of its own. Prefills, joins and the sink layer's step are called eagerly.

A case is a dict with its `kind`, its sizes and a name; `draw` gives others of the same
kinds. Inputs are made on the device from the seed: activations near N(0, 1), weights
scaled so that activations keep that size, quantized words uniform, routed experts
distinct with weights that sum to one.
"""

from __future__ import annotations

import math

import torch

import __graft_entry__

__graft_entry__.load_package()

from mlx_omnia_amd.kernels.add_norm import AddRmsNorm  # noqa: E402
from mlx_omnia_amd.kernels.attention import AttentionStep, FixedKVCache, KVCache  # noqa: E402
from mlx_omnia_amd.kernels.down_combine import DownCombine  # noqa: E402
from mlx_omnia_amd.kernels.gate_up import GateUp  # noqa: E402
from mlx_omnia_amd.kernels.leaf import (QuantizedLinearLeaf, QuantizedSwitchLinearLeaf,  # noqa: E402
                                        RMSNormLeaf, SwiGLU, SwitchLinearLeaf)
from mlx_omnia_amd.kernels.mlp import Mlp  # noqa: E402
from mlx_omnia_amd.kernels.qkv_rope import AngleAtlas, QkvRope, rope_core  # noqa: E402
from mlx_omnia_amd.kernels.route import ResidualRouter, Routing  # noqa: E402
from mlx_omnia_amd.runtime import ops  # noqa: E402

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEVICE = "cuda"
EPS = 1e-6
LAYERS = 4          # layers of a captured decode step
LIMIT = 7.0         # swiglu_oai's clamp
BAND = 128          # rows a sliding layer attends
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def listed() -> list[dict]:
    return [
        # One token's residual join: the smallest call a decode step makes, all latency.
        dict(name="join_decode", kind="join", rows=1, hidden=2048),
        # The same join over a long prompt's rows, of a width that is no power of two.
        dict(name="join_prefill", kind="join", rows=8191, hidden=2880),
        # A prompt's q/k norm and rotation out of the fused projection's rows (Qwen3-4B).
        dict(name="qkv_rope_prefill", kind="qkv_rope", tokens=4096, heads=32, kv_heads=8,
             head_dim=128, pairs=64),
        # A prompt's residual join, router and top-8 (Qwen3-30B-A3B).
        dict(name="router_prefill", kind="router", rows=4096, hidden=2048, experts=128, k=8,
             scoring="softmax", keys=False),
        # Sigmoid routing that hands on logits and ordinal keys, a ragged prompt.
        dict(name="router_keys_ragged", kind="router", rows=1501, hidden=4096, experts=256, k=8,
             scoring="sigmoid", keys=True),
        # A prompt through an attention layer, into an empty cache (Qwen3-30B-A3B).
        dict(name="attention_prefill", kind="prefill", tokens=4096, past=0, heads=32, kv_heads=4,
             head_dim=128, sinks=False, sliding=False),
        # A later chunk of a prompt through a layer with sinks (gpt-oss-120b), odd sizes.
        dict(name="sink_prefill_chunk", kind="prefill", tokens=777, past=1500, heads=64, kv_heads=8,
             head_dim=64, sinks=True, sliding=False),
        # Decode attention over long contexts (Qwen3-4B geometry), four layers.
        dict(name="attention_decode", kind="decode", rows=32768, heads=32, kv_heads=8),
        # One decode step of a layer with sinks over a growing cache (gpt-oss-120b).
        dict(name="sink_step", kind="sink_step", rows=4096, heads=64, kv_heads=8, sliding=False),
        # One token through four layers' routed experts, MXFP4 stacks (gpt-oss-120b).
        dict(name="experts_mxfp4", kind="experts", format="mxfp4", bits=4, group=32, experts=128,
             hidden=2880, inner=2880, slots=4),
        # A prompt chunk's packed down projection with the shared expert (Qwen3-Next-80B-A3B).
        dict(name="shared_down_prefill", kind="shared_down", tokens=512, top_k=10, experts=512,
             hidden=2048),
        # One token through four dense MLPs (Qwen3-4B).
        dict(name="dense_mlp_decode", kind="dense_mlp", hidden=2560, inner=9728),
    ]


def _log(rng, low: int, high: int) -> int:
    """A whole number in [low, high], spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(["join", "qkv_rope", "router", "prefill", "prefill", "decode", "sink_step",
                       "experts", "experts", "shared_down", "dense_mlp"])
    if kind == "join":
        return dict(kind=kind, rows=_log(rng, 1, 8191), hidden=8 * _log(rng, 64, 1024))
    if kind == "qkv_rope":
        head_dim = rng.choice([64, 128, 128, 256])
        kv_heads = rng.choice([2, 4, 8])
        return dict(kind=kind, tokens=_log(rng, 1, 4096), heads=kv_heads * rng.choice([1, 4, 8]),
                    kv_heads=kv_heads, head_dim=head_dim,
                    pairs=rng.choice([head_dim // 2, head_dim // 4]))
    if kind == "router":
        scoring = rng.choice(["softmax", "softmax", "sigmoid"])
        return dict(kind=kind, rows=_log(rng, 1, 4096), hidden=rng.choice([2048, 4096]),
                    experts=rng.choice([128, 256]), k=rng.randint(1, 12), scoring=scoring,
                    keys=scoring == "sigmoid" and rng.random() < 0.5)
    if kind == "prefill":
        sinks = rng.random() < 0.4
        if sinks:
            kv_heads, head_dim, group = rng.choice([4, 8]), 64, 8
        else:
            kv_heads, head_dim, group = rng.choice([2, 4, 8]), 128, rng.choice([1, 2, 4])
        past = 0 if rng.random() < 0.5 else _log(rng, 16, 2500)
        return dict(kind=kind, tokens=_log(rng, 2, 2500), past=past, heads=kv_heads * group,
                    kv_heads=kv_heads, head_dim=head_dim, sinks=sinks,
                    sliding=sinks and rng.random() < 0.5)
    if kind == "decode":
        kv_heads = rng.choice([2, 4, 8])
        return dict(kind=kind, rows=_log(rng, 16, 32768), heads=kv_heads * rng.choice([1, 2, 4, 8]),
                    kv_heads=kv_heads)
    if kind == "sink_step":
        kv_heads = rng.choice([2, 8])
        return dict(kind=kind, rows=_log(rng, 16, 32768), heads=8 * kv_heads, kv_heads=kv_heads,
                    sliding=rng.random() < 0.5)
    if kind == "experts":
        form = rng.choice(["dense", "affine", "affine", "mxfp4", "nvfp4"])
        experts, hidden, inner, slots = rng.choice([
            (128, 2048, 768, 8), (32, 2880, 2880, 4), (64, 2048, 1408, 6), (16, 4096, 1536, 3),
            (8, 1024, 512, 2), (128, 4096, 1536, 8)])
        if form == "affine" and inner > 1536:
            inner = 1440        # the affine down projection takes up to 1536
        if form == "dense" and inner > 2048:
            inner = 1920        # the dense one up to 2048
        bits = rng.choice([2, 3, 4, 4, 5, 6, 8, 8]) if form == "affine" else 4
        # A group has to divide both contractions.
        group = (rng.choice([g for g in (32, 64, 128) if hidden % g == 0 and inner % g == 0])
                 if form == "affine" else {"mxfp4": 32, "nvfp4": 16, "dense": 0}[form])
        return dict(kind=kind, format=form, bits=bits, group=group, experts=experts, hidden=hidden,
                    inner=inner, slots=slots)
    if kind == "shared_down":
        experts = rng.choice([16, 64, 128, 512])
        return dict(kind=kind, tokens=_log(rng, 1, 512), top_k=rng.randint(2, 10), experts=experts,
                    hidden=rng.choice([1024, 1504, 2048]))
    return dict(kind=kind, hidden=8 * _log(rng, 128, 640), inner=8 * _log(rng, 256, 1216))


# Inputs -------------------------------------------------------------------------------


def _make(case: dict, seed: int):
    """(normal, words, generator): seeded makers of device tensors."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(*shape, scale=1.0, shift=0.0, dtype=BF16):
        return (shift + scale * torch.randn(shape, generator=gen, device=DEVICE)).to(dtype)

    def whole(low, high, *shape, dtype=torch.int32):
        return torch.randint(low, high, shape, generator=gen, device=DEVICE, dtype=torch.int32).to(dtype)

    return normal, whole, gen


def _routes(gen, tokens: int, experts: int, k: int):
    """k distinct experts per token and weights that sum to one."""
    scores = torch.rand((tokens, experts), generator=gen, device=DEVICE)
    chosen = torch.topk(scores, k, dim=-1).indices.to(torch.int32).contiguous()
    weights = torch.rand((tokens, k), generator=gen, device=DEVICE) + 0.1
    return chosen, (weights / weights.sum(dim=-1, keepdim=True)).contiguous()


def _stack(case: dict, makers, rows: int, features: int, lead: tuple) -> dict:
    """One projection's expert stack [*lead, rows, features] in the case's format."""
    normal, whole, gen = makers
    form = case.get("format", "nvfp4")
    if form == "dense":
        return dict(weight=normal(*lead, rows, features, scale=features ** -0.5))
    bits = case.get("bits", 4)
    words = whole(-2**31, 2**31 - 1, *lead, rows, features * bits // 32)
    if form == "affine":
        scale = 4.0 / ((1 << bits) * features ** 0.5)
        groups = (*lead, rows, features // case["group"])
        scales = (scale * (0.5 + torch.rand(groups, generator=gen, device=DEVICE))).to(BF16)
        biases = (-scales.float() * ((1 << bits) - 1) / 2).to(BF16)
        return dict(weight=words, scales=scales, biases=biases)
    if form == "mxfp4":
        return dict(weight=words, scales=whole(119, 123, *lead, rows, features // 32, dtype=torch.uint8),
                    bias=normal(*lead, rows, scale=0.25))
    scales = whole(0x08, 0x10, *lead, rows, features // 32, dtype=torch.uint8)
    return dict(weight=words, scales=scales.repeat_interleave(2, dim=-1))


def _leaf(case: dict, stack: dict):
    form = case.get("format", "nvfp4")
    if form == "dense":
        return SwitchLinearLeaf(stack["weight"])
    group, mode = {"affine": (case.get("group"), "affine"), "mxfp4": (32, "mxfp4"),
                   "nvfp4": (16, "nvfp4")}[form]
    kind = QuantizedSwitchLinearLeaf if stack["weight"].dim() == 3 else QuantizedLinearLeaf
    return kind(stack["weight"], stack["scales"], stack.get("biases"), group, case.get("bits", 4), mode=mode)


def _inputs(case: dict, seed: int) -> dict:
    makers = normal, whole, gen = _make(case, seed)
    kind = case["kind"]
    if kind == "join":
        shape = (case["rows"], case["hidden"])
        return dict(x=normal(*shape), branch=normal(*shape),
                    weight=normal(case["hidden"], scale=0.1, shift=1.0))
    if kind == "qkv_rope":
        d = case["head_dim"]
        return dict(fused=normal(1, case["tokens"], (case["heads"] + 2 * case["kv_heads"]) * d),
                    qw=normal(d, scale=0.1, shift=1.0), kw=normal(d, scale=0.1, shift=1.0),
                    offset=int(torch.randint(0, 8192, (1,), generator=gen, device=DEVICE)))
    if kind == "router":
        shape = (case["rows"], case["hidden"])
        return dict(x=normal(*shape), branch=normal(*shape),
                    weight=normal(case["hidden"], scale=0.1, shift=1.0),
                    gate=normal(case["experts"], case["hidden"], scale=0.02),
                    bias=normal(case["experts"], scale=0.1, dtype=F32))
    if kind in ("prefill", "sink_step"):
        d = 64 if kind == "sink_step" else case["head_dim"]
        tokens = 1 if kind == "sink_step" else case["tokens"]
        past = case["rows"] if kind == "sink_step" else case["past"]
        heads, kv = case["heads"], case["kv_heads"]
        got = dict(q=normal(1, tokens, heads * d), k=normal(1, tokens, kv * d), v=normal(1, tokens, kv * d),
                   keys=normal(1, kv, past, d), values=normal(1, kv, past, d), mask="causal")
        if kind == "sink_step" or case["sinks"]:
            got["sinks"] = normal(heads, scale=2.0)
        else:
            got["qw"], got["kw"] = normal(d, scale=0.1, shift=1.0), normal(d, scale=0.1, shift=1.0)
        if case["sliding"]:
            query = past + torch.arange(tokens, device=DEVICE)[:, None]
            row = torch.arange(past + tokens, device=DEVICE)[None]
            got["mask"] = (row <= query) & (row > query - BAND)
        elif tokens == 1:
            got["mask"] = None
        return got
    if kind == "decode":
        heads, kv, rows = case["heads"], case["kv_heads"], case["rows"]
        return dict(layers=[dict(q=normal(heads * 128), k=normal(kv * 128), v=normal(kv * 128),
                                 qw=normal(128, scale=0.1, shift=1.0), kw=normal(128, scale=0.1, shift=1.0),
                                 keys=normal(kv, rows, 128), values=normal(kv, rows, 128))
                            for _ in range(LAYERS)])
    if kind == "experts":
        e, h, i = case["experts"], case["hidden"], case["inner"]
        layers = []
        for _ in range(LAYERS):
            chosen, weights = _routes(gen, 1, e, case["slots"])
            layers.append(dict(x=normal(h), residual=normal(h),
                               chosen=chosen[0].contiguous(), weights=weights[0].contiguous(),
                               up=_stack(case, makers, 2 * i, h, (e,)),
                               down=_stack(case, makers, h, i, (e,))))
        return dict(layers=layers)
    if kind == "shared_down":
        tokens, k, e, h = case["tokens"], case["top_k"], case["experts"], case["hidden"]
        chosen, weights = _routes(gen, tokens, e, k)
        spare = torch.zeros((tokens, 1), dtype=torch.int32, device=DEVICE)
        return dict(act=normal(tokens, k + 1, 512), residual=normal(tokens, h),
                    chosen=torch.cat([chosen, spare], dim=1),
                    weights=torch.cat([weights, spare.to(F32)], dim=1),
                    down=_stack(case, makers, h, 512, (e,)), shared=_stack(case, makers, h, 512, ()))
    h, i = case["hidden"], case["inner"]
    return dict(layers=[dict(x=normal(h), residual=normal(h), up=normal(2 * i, h, scale=h ** -0.5),
                             down=normal(h, i, scale=i ** -0.5)) for _ in range(LAYERS)])


# What a program keeps, and one pass ---------------------------------------------------


def _captured(step) -> dict:
    """`step` captured as a decode loop captures it: a warm-up on a side stream, then the
    graph and the buffers that its replays write."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return dict(graph=graph, out=out)


def prepare(case: dict, seed: int) -> dict:
    inputs = _inputs(case, seed)
    kind = case["kind"]
    state = dict(kind=kind, inputs=inputs)
    if kind == "join":
        state["call"] = AddRmsNorm(RMSNormLeaf(inputs["weight"], EPS),
                                   tokens=1 if case["rows"] == 1 else None)
    elif kind == "qkv_rope":
        state["call"] = QkvRope(
            lambda rows: rows, heads=case["heads"], kv_heads=case["kv_heads"], head_dim=case["head_dim"],
            rope=lambda x, o: rope_core(x, o, base=1e6), eps=EPS, q_norm=inputs["qw"], k_norm=inputs["kw"],
            angles=AngleAtlas(case["pairs"], base=1e6, rows=16384, device=DEVICE),
            rotary_pairs=case["pairs"])
    elif kind == "router":
        bias = inputs["bias"] if case["scoring"] == "sigmoid" else None
        state["call"] = ResidualRouter(
            RMSNormLeaf(inputs["weight"], EPS), inputs["gate"],
            routing=Routing(experts=case["experts"], k=case["k"], scoring=case["scoring"], bias=bias))
        state["keys"] = case["keys"]
    elif kind in ("prefill", "sink_step"):
        d = 64 if kind == "sink_step" else case["head_dim"]
        past = case["rows"] if kind == "sink_step" else case["past"]
        tokens = 1 if kind == "sink_step" else case["tokens"]
        sinks = inputs.get("sinks")
        atlas = AngleAtlas(d // 2, base=150000.0 if sinks is not None else 1e6, rows=past + tokens,
                           device=DEVICE)
        if sinks is not None:
            cache = KVCache()
        else:
            cache = FixedKVCache.empty(case["kv_heads"], past + tokens, d, device=DEVICE)
        if past:
            cache.update_and_fetch(inputs["keys"], inputs["values"])
        state.update(cache=cache, past=past, tokens=tokens, call=AttentionStep(
            cache, heads=case["heads"], kv_heads=case["kv_heads"], head_dim=d, scale=d ** -0.5,
            dtype=BF16, query_weight=inputs.get("qw"), key_weight=inputs.get("kw"), eps=EPS,
            rotary_pairs=d // 2, angles=atlas, sinks=sinks))
    elif kind == "decode":
        heads, kv, rows = case["heads"], case["kv_heads"], case["rows"]
        atlas = AngleAtlas(64, base=1e6, rows=rows, device=DEVICE).atlas
        position = torch.tensor([rows - 1], dtype=torch.int32, device=DEVICE)
        workspace = torch.empty(ops.attention_workspace_bytes(heads, kv, 128, rows), dtype=torch.uint8,
                                device=DEVICE)

        def step():
            outs = [ops.attention_decode(
                one["q"], one["k"], one["v"], one["qw"], one["kw"], atlas, one["keys"], one["values"],
                position, heads=heads, kv_heads=kv, max_rows=rows, scale=128 ** -0.5, eps=EPS,
                workspace=workspace) for one in inputs["layers"]]
            return outs + [one[part][:, rows - 1] for one in inputs["layers"] for part in ("keys", "values")]

        state.update(_captured(step), held=(atlas, position, workspace))
    elif kind == "experts":
        form, h, i = case["format"], case["hidden"], case["inner"]
        layout = "blocked" if form == "dense" else "interleaved"
        pairs = []
        for one in inputs["layers"]:
            oai = dict(activation="swiglu_oai", limit=LIMIT, bias=one["up"].get("bias")) if form == "mxfp4" else {}
            pairs.append((GateUp(_leaf(case, one["up"]), hidden=h, inner=i, layout=layout, **oai),
                          DownCombine(_leaf(case, one["down"]), hidden=h, inner=i, layout=layout,
                                      bias=one["down"].get("bias"))))

        def step():
            return [down(up(one["x"], one["chosen"]), one["chosen"], one["weights"], one["residual"])
                    for one, (up, down) in zip(inputs["layers"], pairs)]

        state.update(_captured(step), held=pairs)
    elif kind == "shared_down":
        state["call"] = DownCombine(_leaf(case, inputs["down"]), hidden=case["hidden"], inner=512,
                                    shared=_leaf(case, inputs["shared"]))
    else:
        mlps = []
        for one in inputs["layers"]:
            leaf = SwiGLU(8, 8)
            leaf.gate_up_proj.weight = torch.nn.Parameter(one["up"], requires_grad=False)
            leaf.down_proj.weight = torch.nn.Parameter(one["down"], requires_grad=False)
            mlps.append(Mlp(leaf, hidden=case["hidden"], inner=case["inner"]))

        def step():
            return [mlp(one["x"], one["residual"]) for one, mlp in zip(inputs["layers"], mlps)]

        state.update(_captured(step), held=mlps)
    return state


def run(state: dict):
    kind, inputs = state["kind"], state["inputs"]
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    call = state["call"]
    if kind == "join":
        return call(inputs["x"], inputs["branch"])
    if kind == "qkv_rope":
        return call(inputs["fused"], inputs["offset"])
    if kind == "router":
        if state["keys"]:
            summed, normalized, logits, keys = call.with_keys(inputs["x"], inputs["branch"])
            return summed, normalized, logits, keys.view(torch.int32)
        return call(inputs["x"], inputs["branch"])
    if kind in ("prefill", "sink_step"):
        # A new request takes the cache over from `past` rows on.
        cache, past = state["cache"], state["past"]
        cache.offset = past
        if isinstance(cache, FixedKVCache):
            cache.position.fill_(past)
        out = call(inputs["q"], inputs["k"], inputs["v"], inputs["mask"])
        rows = slice(past, past + state["tokens"])
        return out, cache.keys[:, :, rows], cache.values[:, :, rows]
    return call(inputs["act"], inputs["chosen"], inputs["weights"], inputs["residual"])


# What a pass cannot do without --------------------------------------------------------


def _attended(case: dict) -> int:
    """Pairs of a query and a row that it attends, for one head."""
    tokens, past = case["tokens"], case["past"]
    if case["sliding"]:
        return sum(min(BAND, past + t + 1) for t in range(tokens))
    return tokens * past + tokens * (tokens + 1) // 2


def _row_bytes(case: dict, features: int) -> float:
    form = case.get("format", "nvfp4")
    return {"dense": 2 * features, "mxfp4": features / 2 + features / 32 + 2,
            "nvfp4": features / 2 + features / 16}.get(
                form) or features * case["bits"] / 8 + 4 * features / case["group"]


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "join":
        return dict(bytes=8 * case["rows"] * case["hidden"] + 2 * case["hidden"],
                    flops=6 * case["rows"] * case["hidden"])
    if kind == "qkv_rope":
        values = case["tokens"] * (case["heads"] + case["kv_heads"]) * case["head_dim"]
        return dict(bytes=4 * values + 8 * case["pairs"] * case["tokens"], flops=10 * values)
    if kind == "router":
        rows, h, e = case["rows"], case["hidden"], case["experts"]
        out = 6 * e if case["keys"] else 8 * case["k"]
        return dict(bytes=8 * rows * h + 2 * e * h + rows * out, flops=2 * rows * h * e)
    if kind == "prefill":
        d, heads, kv = case["head_dim"], case["heads"], case["kv_heads"]
        rows = case["past"] + case["tokens"]
        if case["sliding"]:
            rows = min(rows, case["tokens"] + BAND)
        return dict(bytes=4 * case["tokens"] * heads * d + 4 * kv * d * (rows + 2 * case["tokens"]),
                    flops=4 * _attended(case) * heads * d)
    if kind == "sink_step":
        rows = min(case["rows"] + 1, BAND) if case["sliding"] else case["rows"] + 1
        return dict(bytes=4 * case["kv_heads"] * 64 * rows + 4 * case["heads"] * 64,
                    flops=4 * rows * case["heads"] * 64)
    if kind == "decode":
        rows, heads, kv = case["rows"], case["heads"], case["kv_heads"]
        return dict(bytes=LAYERS * (4 * kv * 128 * (rows + 2) + 4 * heads * 128),
                    flops=LAYERS * 4 * rows * heads * 128)
    if kind == "experts":
        h, i, s = case["hidden"], case["inner"], case["slots"]
        weights = s * (2 * i * _row_bytes(case, h) + h * _row_bytes(case, i))
        return dict(bytes=LAYERS * (weights + 4 * h), flops=LAYERS * 6 * s * i * h)
    if kind == "shared_down":
        tokens, slots, h = case["tokens"], case["top_k"] + 1, case["hidden"]
        stacks = min(case["experts"], tokens * case["top_k"]) + 1
        return dict(bytes=stacks * h * _row_bytes(case, 512) + 2 * tokens * slots * 512 + 4 * tokens * h,
                    flops=2 * tokens * slots * 512 * h)
    h, i = case["hidden"], case["inner"]
    return dict(bytes=LAYERS * (6 * h * i + 4 * h), flops=LAYERS * 6 * h * i)


def tolerance(case: dict) -> dict:
    """bf16 results: about four times the distance of each path from its 64-bit values."""
    return {"rel": 1e-2, "max": 0.1}


# The same results in 64 bits ----------------------------------------------------------


def _norm64(x, weight):
    return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + EPS) * weight.to(F64)


def _rotate64(x, first: int, pairs: int, base: float):
    """[..., T, D] at positions first .. first + T - 1."""
    index = torch.arange(pairs, dtype=F64, device=x.device)
    positions = torch.arange(first, first + x.shape[-2], dtype=F64, device=x.device)
    theta = positions[:, None] * torch.exp(-math.log(base) * index / pairs)[None]
    cos, sin = torch.cos(theta), torch.sin(theta)
    a, b = x[..., :pairs], x[..., pairs : 2 * pairs]
    return torch.cat([a * cos - b * sin, a * sin + b * cos, x[..., 2 * pairs :]], dim=-1)


def _attend64(q, keys, values, scale, allowed, sinks):
    """q [H, T, D] over keys, values [KV, R, D], a few heads at a time."""
    heads, group, outs = q.shape[0], q.shape[0] // keys.shape[0], []
    for h in range(heads):
        k, v = keys[h // group], values[h // group]
        s = torch.matmul(q[h], k.t().contiguous()) * scale
        if allowed is not None:
            s = s.masked_fill(~allowed, float("-inf"))
        if sinks is not None:
            s = torch.cat([sinks[h].expand(s.shape[0], 1), s], dim=-1)
            outs.append(torch.matmul(torch.softmax(s, dim=-1)[:, 1:], v))
        else:
            outs.append(torch.matmul(torch.softmax(s, dim=-1), v))
    return torch.stack(outs)


def _matrix64(case: dict, stack: dict, pick=None):
    """A stack's matrices (those picked) in 64 bits."""
    take = (lambda t: t) if pick is None else (lambda t: t[pick.long()])
    weight = take(stack["weight"])
    form = case.get("format", "nvfp4")
    if form == "dense":
        return weight.to(F64)
    bits = case.get("bits", 4)
    words = weight.to(torch.int64) & 0xFFFFFFFF
    bit = torch.arange(words.shape[-1] * 32 // bits, device=DEVICE) * bits
    spare = torch.cat([words, torch.zeros_like(words[..., :1])], dim=-1)
    codes = ((spare[..., bit // 32] | (spare[..., bit // 32 + 1] << 32)) >> (bit % 32)) & ((1 << bits) - 1)
    scales = take(stack["scales"])
    if form == "affine":
        group = case["group"]
        return (codes.to(F64) * scales.to(F64).repeat_interleave(group, dim=-1)
                + take(stack["biases"]).to(F64).repeat_interleave(group, dim=-1))
    values = torch.tensor(E2M1, dtype=F64, device=DEVICE)[codes]
    if form == "mxfp4":
        return values * torch.exp2(scales.to(F64) - 127).repeat_interleave(32, dim=-1)
    exponent, mantissa = (scales.to(torch.int64) >> 3) & 15, (scales.to(torch.int64) & 7).to(F64)
    factor = torch.where(exponent > 0, (1 + mantissa / 8) * torch.exp2(exponent.to(F64) - 7), mantissa * 2.0 ** -9)
    return values * factor.repeat_interleave(16, dim=-1)


def exact(case: dict, seed: int):
    inputs = _inputs(case, seed)
    kind = case["kind"]
    if kind == "join":
        summed = (inputs["x"].to(F64) + inputs["branch"].to(F64)).to(BF16).to(F64)
        return summed, _norm64(summed, inputs["weight"])
    if kind == "qkv_rope":
        d, heads, kv = case["head_dim"], case["heads"], case["kv_heads"]
        rows = inputs["fused"][0].to(F64).unflatten(-1, (heads + 2 * kv, d)).transpose(0, 1)
        turn = lambda part, w: _rotate64(_norm64(part, w), inputs["offset"], case["pairs"], 1e6)[None]  # noqa: E731
        return (turn(rows[:heads], inputs["qw"]), turn(rows[heads : heads + kv], inputs["kw"]),
                rows[heads + kv :][None])
    if kind == "router":
        # The join, the norm and the logits are bf16 values by declaration.
        summed = (inputs["x"].to(F64) + inputs["branch"].to(F64)).to(BF16).to(F64)
        normalized = _norm64(summed, inputs["weight"])
        logits = normalized.to(BF16).to(F64) @ inputs["gate"].to(F64).t().contiguous()
        if case["keys"]:
            return summed, normalized, logits, None
        return summed, normalized, None, None
    if kind in ("prefill", "sink_step"):
        d = 64 if kind == "sink_step" else case["head_dim"]
        tokens = 1 if kind == "sink_step" else case["tokens"]
        past = case["rows"] if kind == "sink_step" else case["past"]
        heads, kv, sinks = case["heads"], case["kv_heads"], inputs.get("sinks")
        split = lambda t, n: t[0].to(F64).unflatten(-1, (n, d)).transpose(0, 1)  # noqa: E731
        q, k, v = split(inputs["q"], heads), split(inputs["k"], kv), split(inputs["v"], kv)
        if sinks is None:
            q, k = _norm64(q, inputs["qw"]), _norm64(k, inputs["kw"])
        base = 1e6 if sinks is None else 150000.0
        q, k = _rotate64(q, past, d // 2, base), _rotate64(k, past, d // 2, base)
        keys = torch.cat([inputs["keys"][0].to(F64), k], dim=1)
        values = torch.cat([inputs["values"][0].to(F64), v], dim=1)
        allowed = inputs["mask"]
        if isinstance(allowed, str):
            query = past + torch.arange(tokens, device=DEVICE)[:, None]
            allowed = torch.arange(past + tokens, device=DEVICE)[None] <= query
        out = _attend64(q, keys, values, d ** -0.5, allowed, None if sinks is None else sinks.to(F64))
        return out[None], k[None], v[None]
    if kind == "decode":
        heads, kv, last = case["heads"], case["kv_heads"], case["rows"] - 1
        outs, written = [], []
        for one in inputs["layers"]:
            q = _rotate64(_norm64(one["q"].to(F64).reshape(heads, 1, 128), one["qw"]), last, 64, 1e6)
            k = _rotate64(_norm64(one["k"].to(F64).reshape(kv, 1, 128), one["kw"]), last, 64, 1e6)
            v = one["v"].to(F64).reshape(kv, 1, 128)
            keys = torch.cat([one["keys"][:, :last].to(F64), k], dim=1)
            values = torch.cat([one["values"][:, :last].to(F64), v], dim=1)
            outs.append(_attend64(q, keys, values, 128 ** -0.5, None, None)[:, 0])
            written += [k[:, 0], v[:, 0]]
        return outs + written
    if kind == "experts":
        outs = []
        for one in inputs["layers"]:
            r = _matrix64(case, one["up"], one["chosen"]) @ one["x"].to(F64)
            if case["format"] == "mxfp4":
                r = r + one["up"]["bias"][one["chosen"].long()].to(F64)
            if case["format"] == "dense":
                gate, up = r.chunk(2, dim=-1)
            else:
                gate, up = r[:, 0::2], r[:, 1::2]
            if case["format"] == "mxfp4":
                gate, up = gate.clamp(max=LIMIT), up.clamp(-LIMIT, LIMIT)
                act = gate * torch.sigmoid(1.702 * gate) * (up + 1)
            else:
                act = gate * torch.sigmoid(gate) * up
            d = torch.matmul(_matrix64(case, one["down"], one["chosen"]), act[..., None])[..., 0]
            if case["format"] == "mxfp4":
                d = d + one["down"]["bias"][one["chosen"].long()].to(F64)
            outs.append(one["residual"].to(F64) + (d * one["weights"].to(F64)[:, None]).sum(dim=0))
        return outs
    if kind == "shared_down":
        act, k = inputs["act"].to(F64), case["top_k"]
        out = inputs["residual"].to(F64) + act[:, k] @ _matrix64(case, inputs["shared"]).t().contiguous()
        for expert in torch.unique(inputs["chosen"][:, :k]).tolist():
            token, slot = torch.nonzero(inputs["chosen"][:, :k] == expert, as_tuple=True)
            matrix = _matrix64(case, inputs["down"], torch.tensor([expert], device=DEVICE))[0]
            part = act[token, slot] @ matrix.t().contiguous()
            out.index_add_(0, token, part * inputs["weights"][token, slot].to(F64)[:, None])
        return out
    outs = []
    for one in inputs["layers"]:
        gate, up = (one["up"].to(F64) @ one["x"].to(F64)).chunk(2)
        outs.append(one["residual"].to(F64) + one["down"].to(F64) @ (gate * torch.sigmoid(gate) * up))
    return outs
