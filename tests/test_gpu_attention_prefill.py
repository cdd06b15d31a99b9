"""The prefill kernels (csrc/attention_prefill.hip) against the Core chain on the same device.

Sizes straddle the kernel's tiles (32 queries a wave, 64 rows a tile), every way a
workgroup's waves split into heads and queries, both head widths, causal, unmasked and
boolean masks, with and without sinks, gains, rotation and earlier rows.

Bar: the bf16 bar (assert_bf16_close), at least 98% of the context bit-identical to the
fp32 Core chain (both round once from fp32 sums of the same products in another order: a
value flips where the sums' difference, about sqrt(rows) 2^-24 of it, crosses a rounding
point, so well under 1% do); the cache rows likewise at 99.9%, values bit-exact.
"""

import numpy as np
import pytest
import torch

from mlx_omnia_amd.kernels.resolve import FALLBACKS
from mlx_omnia_amd.kernels.attention import AttentionStep, FixedKVCache, KVCache
from mlx_omnia_amd.kernels.qkv_rope import AngleAtlas, AngleTable
from mlx_omnia_amd.runtime import ops
from util import assert_bf16_close, bits_of

pytestmark = pytest.mark.gpu


class Layer:
    """Two steps over equal caches: the binding's and the Core chain's."""

    def __init__(self, seed, heads, kv_heads, d, past, tokens, *, sinks=False, gains=True, pairs=None,
                 mscale=1.0, growing=None, angles=None):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        self.normal = lambda *shape, s=1.0, m=0.0: (
            m + s * torch.randn(shape, generator=gen, device="cuda")).to(torch.bfloat16)
        pairs = d // 2 if pairs is None else pairs
        sink = self.normal(heads, s=2.0) if sinks else None
        declare = dict(heads=heads, kv_heads=kv_heads, head_dim=d, scale=d ** -0.5, dtype=torch.bfloat16,
                       rotary_pairs=pairs, mscale=mscale, sinks=sink,
                       angles=angles or AngleAtlas(pairs, base=1e4, rows=past + tokens + 8, device="cuda"))
        if gains:
            declare.update(query_weight=self.normal(d, s=0.1, m=1.0), key_weight=self.normal(d, s=0.1, m=1.0))
        keys, values = self.normal(1, kv_heads, past, d), self.normal(1, kv_heads, past, d)
        self.caches, self.steps = [], []
        for reference in (False, True):
            cache = KVCache() if sinks else FixedKVCache.empty(kv_heads, past + tokens + 3, d, device="cuda")
            if past:
                cache.update_and_fetch(keys, values)
            self.caches.append(cache)
            self.steps.append(AttentionStep(cache, reference=reference, **declare))
        self.raw = [self.normal(1, tokens, n * d) for n in (heads, kv_heads, kv_heads)]
        self.past, self.tokens = past, tokens

    def check(self, mask, raw=None, fallbacks=0):
        raw = raw or self.raw
        before = sum(FALLBACKS.values())
        got = self.steps[0](*raw, mask=mask)
        assert sum(FALLBACKS.values()) == before + fallbacks
        want = self.steps[1](*raw, mask=mask)
        assert got.shape == want.shape and got.is_contiguous()
        assert_bf16_close(bits_of(got), bits_of(want), min_exact=0.98)
        ours, core = self.caches
        assert ours.offset == core.offset == self.past + self.tokens
        if isinstance(ours, FixedKVCache):
            assert int(ours.position.item()) == ours.offset
        assert ours.keys.shape == core.keys.shape
        assert_bf16_close(bits_of(ours.keys), bits_of(core.keys), min_exact=0.999)
        assert torch.equal(ours.values, core.values)
        return got


@pytest.mark.parametrize("tokens,past", [(2, 0), (31, 0), (32, 1), (33, 31), (64, 0), (65, 63), (129, 64),
                                         (300, 77), (7, 1000)])
@pytest.mark.parametrize("heads,kv_heads", [(2, 2), (4, 2), (8, 2), (8, 1)])
def test_causal_prefill_matches_the_core_chain(tokens, past, heads, kv_heads):
    print(f"prefill d=128 H={heads}/{kv_heads} T={tokens} past={past}", flush=True)
    Layer(tokens + past, heads, kv_heads, 128, past, tokens).check("causal")


@pytest.mark.parametrize("tokens,past", [(2, 0), (33, 100), (64, 64), (200, 0)])
@pytest.mark.parametrize("mask", ["causal", "band", None])
def test_sink_prefill_matches_the_core_chain(tokens, past, mask):
    print(f"prefill sinks T={tokens} past={past} mask={mask}", flush=True)
    layer = Layer(tokens + past + 1, 16, 2, 64, past, tokens, sinks=True, gains=False)
    if mask == "band":
        query = past + torch.arange(tokens, device="cuda")[:, None]
        row = torch.arange(past + tokens, device="cuda")[None]
        mask = ((row <= query) & (row > query - 40))[None, None]
        mask[:, :, 0] = False     # the first query attends the sink alone: zeros
    got = layer.check(mask)
    if torch.is_tensor(mask):
        assert not bool(got[0, :, 0].any())


@pytest.mark.parametrize("tokens,past,heads,kv_heads,sinks", [
    (2, 1000, 4, 4, False), (5, 2111, 8, 1, False), (70, 600, 2, 2, False), (3, 900, 8, 2, True),
    (40, 5000, 16, 2, True),
])
@pytest.mark.parametrize("banded", [False, True])
def test_keys_walked_by_several_workgroups(tokens, past, heads, kv_heads, sinks, banded):
    """Short prompts over many rows: the splits' states merged, with bands that leave whole
    splits, whole windows of 64 tiles and whole queries without a row (masks of odd strides)."""
    print(f"prefill splits H={heads}/{kv_heads} T={tokens} past={past} sinks={sinks} banded={banded}", flush=True)
    assert ops.library().omnia_attention_prefill_workspace_bytes(
        heads, kv_heads, 64 if sinks else 128, tokens, past + tokens) > 0
    layer = Layer(tokens + past, heads, kv_heads, 64 if sinks else 128, past, tokens, sinks=sinks, gains=not sinks)
    mask = "causal"
    if banded:
        query = past + torch.arange(tokens, device="cuda")[:, None]
        row = torch.arange(past + tokens, device="cuda")[None]
        wide = torch.zeros((tokens, past + tokens + 5), dtype=torch.bool, device="cuda")
        wide[:, 3 : 3 + past + tokens] = ((row <= query) & (row > query - 100)) | (row == 7)
        if sinks:
            wide[1] = False
        mask = wide[:, 3 : 3 + past + tokens]
    layer.check(mask)


def test_partial_rotation_factor_and_strided_rows():
    layer = Layer(5, 8, 2, 128, 20, 50, pairs=32, mscale=1.3465735912322998)
    fused = layer.normal(1, 50, 12 * 128)   # q, k and v as slices of one projection's rows
    layer.check("causal", raw=[fused[..., :1024], fused[..., 1024:1280], fused[..., 1280:]])
    table = AngleTable(*(torch.rand(64, 64, device="cuda") for _ in range(2)))
    Layer(6, 4, 4, 128, 3, 40, angles=table).check(None)


def test_calls_the_kernels_do_not_compute_stay_with_the_core_chain():
    layer = Layer(7, 4, 2, 128, 10, 40)
    additive = torch.zeros((40, 50), device="cuda")
    layer.check(additive, fallbacks=1)
    layer = Layer(8, 4, 2, 128, 10, 40)
    raw = [layer.raw[0].clone().requires_grad_(), *layer.raw[1:]]
    step = layer.steps[0]
    out = step(*raw, mask="causal")
    assert out.requires_grad
    short = AngleTable(*(torch.rand(20, 64, device="cuda") for _ in range(2)))
    with pytest.raises(RuntimeError):      # the table ends before the prompt does
        Layer(9, 4, 2, 128, 0, 40, angles=short).steps[0](*layer.raw, mask="causal")
    cache = layer.caches[1]
    with pytest.raises(ValueError):
        layer.steps[0](*layer.raw, mask="causal")   # the cache is full
    assert cache.offset == 10


def test_a_row_that_attends_nothing_is_nan_and_later_rows_are_not_read():
    layer = Layer(10, 4, 2, 128, 0, 70)
    mask = torch.ones((70, 70), dtype=torch.bool, device="cuda").tril()
    mask[66] = False
    got, want = (step(*layer.raw, mask=mask) for step in layer.steps)
    assert torch.equal(got.isnan(), want.isnan()) and bool(got[0, :, 66].isnan().all())
    keep = ~want.isnan()
    assert_bf16_close(bits_of(got[keep]), bits_of(want[keep]), min_exact=0.98)
    cache = layer.caches[0]
    cache.keys[:, :, 70:], cache.values[:, :, 70:] = float("nan"), float("inf")
    cache.offset = 0
    again = layer.steps[0](*layer.raw, mask=mask)
    assert np.array_equal(bits_of(got), bits_of(again))


@pytest.mark.parametrize("past,tokens", [(0, 70), (300, 5)])
def test_an_infinite_value_gives_that_infinity(past, tokens):
    layer = Layer(12, 8, 2, 128, past, tokens)
    plain = layer.steps[0](*layer.raw, mask=None)
    layer.caches[0].offset = past
    raw = [layer.raw[0], layer.raw[1], layer.raw[2].clone()]
    row = raw[2].view(tokens, -1)[2]
    row[5], row[77] = float("inf"), float("-inf")      # the first cached head's
    got = layer.steps[0](*raw, mask=None)
    rest = [d for d in range(128) if d not in (5, 77)]
    assert bool((got[:, :4, :, 5] == float("inf")).all()) and bool((got[:, :4, :, 77] == float("-inf")).all())
    assert torch.equal(got[..., rest], plain[..., rest]) and torch.equal(got[:, 4:], plain[:, 4:])


@pytest.mark.parametrize("past,tokens,d", [(0, 65, 128), (0, 127, 64), (300, 5, 128), (600, 5, 128), (900, 3, 64)])
def test_an_infinite_value_in_the_last_row(past, tokens, d):
    """The last tile ends past the last row: what stands there in its place has no part in
    the products (with one workgroup over the keys and with several)."""
    print(f"prefill infinite last row D={d} T={tokens} past={past}", flush=True)
    assert (past + tokens) % 64
    layer = Layer(13, 8, 2, d, past, tokens, sinks=d == 64, gains=d == 128)
    plain = layer.steps[0](*layer.raw, mask=None)
    layer.caches[0].offset = past
    raw = [layer.raw[0], layer.raw[1], layer.raw[2].clone()]
    row = raw[2].view(tokens, -1)[-1]
    row[5], row[d + 40] = float("inf"), float("-inf")      # of either cached head
    got = layer.steps[0](*raw, mask=None)
    assert bool((got[:, :4, :, 5] == float("inf")).all()) and bool((got[:, 4:, :, 40] == float("-inf")).all())
    plain[:, :4, :, 5], plain[:, 4:, :, 40] = float("inf"), float("-inf")
    assert torch.equal(got, plain)


@pytest.mark.parametrize("past,tokens", [(0, 40), (900, 3)])
def test_sinks_that_are_not_finite(past, tokens):
    """As the softmax over the logits has them: one of -inf has no weight (and a query that
    attends nothing else no result), one of +inf or NaN leaves no result, a huge one zeros."""
    print(f"prefill sinks not finite T={tokens} past={past}", flush=True)
    layer = Layer(14, 8, 2, 64, past, tokens, sinks=True, gains=False)
    for head, value in ((0, float("-inf")), (1, -3.3e38), (2, 3.3e38), (3, float("inf")), (5, float("nan"))):
        layer.steps[0].strategy.sinks[head] = value
    assert layer.steps[1].strategy.sinks.data_ptr() == layer.steps[0].strategy.sinks.data_ptr()
    mask = torch.ones((tokens, past + tokens), dtype=torch.bool, device="cuda").tril(past)
    mask[1] = False
    got, want = (step(*layer.raw, mask=mask) for step in layer.steps)
    assert torch.equal(got.isnan(), want.isnan())
    assert bool(want[0, 0, 1].isnan().all()) and bool(want[0, [3, 5]].isnan().all())
    assert not bool(want[0, 0, 2:].isnan().any()) and not bool(want[0, 2].any())
    assert not bool(want[0, 1, 1].any())
    keep = ~want.isnan()
    assert_bf16_close(bits_of(got[keep]), bits_of(want[keep]), min_exact=0.98)
