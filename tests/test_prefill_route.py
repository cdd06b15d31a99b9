"""Which calls the prefill kernels take, on the CPU: the device gate is held open and the two
kernels replaced by stand-ins that no tracer, transform or compiler can see into (as the real
ones), so that a call that one of these follows shows which way it went.
"""

import importlib

import pytest
import torch

from mlx_omnia_amd.kernels.attention import DefaultAttentionStep, FixedKVCache, HipAttentionStep
from mlx_omnia_amd.kernels.qkv_rope import AngleAtlas, AngleTable

route = importlib.import_module("mlx_omnia_amd.kernels.attention.prefill")
HEADS, KV_HEADS, D, TOKENS = 4, 2, 128, 5


@pytest.fixture
def kernels(monkeypatch):
    """The names of the kernels that were reached."""
    reached = []

    def project(raw_queries, raw_keys, raw_values, *rest, heads, head_dim, **_):
        reached.append("project")
        return torch.zeros((heads, raw_queries.shape[1], head_dim), dtype=torch.bfloat16)

    def attention(queries, keys, values, **_):
        reached.append("prefill")
        return torch.zeros(queries.shape, dtype=torch.bfloat16)

    monkeypatch.setattr(route, "hip_device", lambda *tensors: True)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: -1, raising=False)
    monkeypatch.setattr(route.ops, "attention_project", project)
    monkeypatch.setattr(route.ops, "attention_prefill", attention)
    return reached


def rows(seed, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def raw_rows(seed):
    return [rows(seed + i, 1, TOKENS, n * D) for i, n in enumerate((HEADS, KV_HEADS, KV_HEADS))]


def layer(*, angles=None, query_gain=None, past=0, capacity=64):
    """(the step with the kernels, the Core chain over a cache of its own)"""
    steps = []
    angles = angles or AngleAtlas(D // 2, base=1e4, rows=64)
    gains = (rows(1, D) if query_gain is None else query_gain, rows(2, D))
    for _ in range(2):
        cache = FixedKVCache.empty(KV_HEADS, capacity, D)
        if past:
            cache.update_and_fetch(rows(3, 1, KV_HEADS, past, D), rows(4, 1, KV_HEADS, past, D))
        core = DefaultAttentionStep.build(
            cache, heads=HEADS, kv_heads=KV_HEADS, head_dim=D, scale=D ** -0.5, dtype=torch.bfloat16,
            query_weight=gains[0], key_weight=gains[1], eps=1e-6, rotary_pairs=D // 2, mscale=1.0,
            angles=angles, base=1e4, sinks=None)
        steps.append(core)
    core = steps[0]
    step = HipAttentionStep(core.cache, HEADS, KV_HEADS, core.scale, core.eps, 1.0, core.query_weight,
                            core.key_weight, torch.empty(0), None, torch.empty(0), core)
    return step, steps[1]


def test_a_plain_call_takes_the_kernels(kernels):
    step, _ = layer()
    step(*raw_rows(10), mask="causal")
    assert kernels == ["project", "prefill"] and step.cache.offset == TOKENS


def test_a_traced_call_replays_on_new_inputs(kernels):
    step, core = layer()
    traced = torch.jit.trace(lambda *raw: step(*raw, mask="causal"), tuple(raw_rows(10)), check_trace=False)
    assert kernels == []
    fresh = raw_rows(20)
    assert torch.equal(traced(*fresh), core(*fresh, mask="causal"))


def test_a_compiled_call_is_one_graph_of_the_core_chain(kernels):
    step, core = layer()
    raw = raw_rows(10)
    compiled = torch.compile(lambda *raw: step(*raw, mask="causal"), backend="eager", fullgraph=True)
    assert torch.equal(compiled(*raw), core(*raw, mask="causal"))
    assert kernels == [] and step.cache.offset == TOKENS


def test_a_gain_that_a_transform_follows(kernels):
    raw = raw_rows(10)

    def loss(gain, steps):
        return layer(query_gain=gain)[steps](*raw, mask="causal").float().square().sum()

    got, want = (torch.func.grad(loss)(rows(1, D), steps) for steps in (0, 1))
    assert kernels == [] and bool(want.any()) and torch.equal(got, want)


@pytest.mark.parametrize("table", ["table", "callable"])
def test_angles_with_a_gradient(kernels, table):
    raw = raw_rows(10)
    theta = torch.arange(64.0)[:, None] * torch.linspace(1.0, 0.1, D // 2)
    gradients = []
    for index in (0, 1):
        scale = torch.ones((), requires_grad=True)
        cos, sin = torch.cos(theta * scale), torch.sin(theta * scale)
        angles = (AngleTable(cos, sin) if table == "table"
                  else lambda offset, length: torch.cat([cos, sin], dim=-1)[offset : offset + length])
        layer(angles=angles)[index](*raw, mask="causal").float().square().sum().backward()
        gradients.append(scale.grad)
    assert kernels == [] and bool(gradients[1] != 0) and torch.equal(*gradients)


@pytest.mark.parametrize("heads,capacity", [(8192, 8), (1, 1 << 24)])
def test_sizes_past_the_kernels_stay_with_the_core_chain(kernels, heads, capacity):
    """Seen before anything is written: the entries themselves would refuse the attention
    after the prologue had written the cache."""
    cache = FixedKVCache(*(torch.empty((1, 1, capacity, 64), dtype=torch.bfloat16) for _ in range(2)),
                         position=capacity - 2)
    core = DefaultAttentionStep.build(
        cache, heads=heads, kv_heads=1, head_dim=64, scale=0.125, dtype=torch.bfloat16, query_weight=None,
        key_weight=None, eps=1e-6, rotary_pairs=0, mscale=1.0, angles=None, base=1e4, sinks=None)
    raw = [rows(30, 1, 2, n * 64) for n in (heads, 1, 1)]
    assert route.prefill(core, *raw, "causal") is None
    assert kernels == [] and cache.offset == capacity - 2
    lib = route.ops.library()
    assert lib.omnia_attention_prefill_workspace_bytes(heads, 1, 64, 2, capacity) < 0
    assert lib.omnia_attention_prefill_workspace_bytes(min(heads, 4096), 1, 64, 2, capacity - 1) >= 0


def test_a_gain_of_another_shape_is_refused_as_before(kernels):
    raw = raw_rows(10)
    for index in (0, 1):
        step = layer(query_gain=rows(1, D, 1))[index]
        with pytest.raises(RuntimeError):     # D values, but not along the head
            step(*raw, mask="causal")
    step, core = layer(query_gain=rows(1, 1, D))
    step(*raw, mask="causal")
    assert kernels == ["project", "prefill"]
