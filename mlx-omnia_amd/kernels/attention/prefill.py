"""A prefill (or one step of a sink layer) on `omnia_attention_project` and
`omnia_attention_prefill` (csrc/attention_prefill.hip): the norms, the rotation, the cache
write and the attention that `DefaultAttentionStep` runs in torch ops
(core/kernels/attention/default.py:85-156), for the calls these kernels compute alike.

`project_served` says whether a call's prologue is one of them, before anything is written:
plain bf16 tensors of the current ROCm device, head_dim 64 or 128, a cache of this package
with room, gains and angle rows the kernel can read. A call that autograd, a functorch
transform, a dispatch mode, a tracer or a compiler follows stays with the torch ops, which
they can see through. `mask_served` does the same for the attention's mask.
"""

from __future__ import annotations

import math

import torch
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from ...runtime import ops
from .._device import hip_device
from ..qkv_rope.atlas import AngleAtlas
from ..qkv_rope.kernel import AngleTable
from .cache import FixedKVCache, KVCache

HEAD_DIMS = (64, 128)
MAX_HEADS, MAX_ROWS = 4096, 1 << 24   # what the entries take: as many heads, fewer rows
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def plain_call(*tensors: torch.Tensor) -> bool:
    """Ordinary tensors on the current ROCm device, with nothing following the operations
    on them: a kernel may then stand in for torch ops."""
    # First, since a compiler follows the questions below as well.
    if torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None:
        return False
    if torch._C._len_torch_dispatch_stack():
        return False
    if torch._C._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0:
        return False
    if torch._C._len_torch_function_stack() and any(
            type(mode) is not DeviceContext for mode in _get_current_function_mode_stack()):
        return False
    followed, index = torch.is_grad_enabled(), tensors[0].get_device()
    for t in tensors:
        if type(t) not in _PLAIN or t.get_device() != index or (followed and t.requires_grad):
            return False
    return hip_device(tensors[0]) and index == torch._C._cuda_getDevice()


def _gain_readable(weight: torch.Tensor | None, head_dim: int) -> bool:
    return weight is None or (weight.dtype == torch.bfloat16 and weight.is_contiguous()
                              and weight.numel() == head_dim == weight.shape[-1]
                              and weight.data_ptr() % 16 == 0)


def _cache_writable(cache, length: int, kv_heads: int, head_dim: int) -> bool:
    """A cache whose rows the prologue may write itself: a fixed one with room, or a growing
    one, of bf16 rows the kernels read in place."""
    if type(cache) is FixedKVCache and cache.offset + length > cache.capacity:
        return False
    for buffer in (cache.keys, cache.values):
        if buffer is None:
            continue
        if buffer.dtype != torch.bfloat16 or buffer.dim() != 4 or not buffer.is_contiguous():
            return False
        lead, heads, _, width = buffer.shape
        if lead != 1 or heads != kv_heads or width != head_dim or buffer.data_ptr() % 16 != 0:
            return False
    return True


def project_served(core, raw_queries, raw_keys, raw_values) -> bool:
    """Whether `project` computes this call's prologue as `core` (a `DefaultAttentionStep`)
    does."""
    d, cache = core.head_dim, core.cache
    if type(cache) is not KVCache and type(cache) is not FixedKVCache:
        return False
    held = [t for t in (core.query_weight, core.key_weight, core.sinks, cache.keys, cache.values) if t is not None]
    # Ahead of the questions about addresses, which a wrapped tensor does not answer.
    if not plain_call(raw_queries, raw_keys, raw_values, *held):
        return False
    if raw_queries.dim() != 3 or d not in HEAD_DIMS or core.heads % core.kv_heads or core.heads > MAX_HEADS:
        return False
    length = raw_queries.shape[1]
    rows = (1, length, core.kv_heads * d)
    if (length == 0 or raw_queries.shape != (1, length, core.heads * d) or raw_keys.shape != rows
            or raw_values.shape != rows):
        return False
    if not raw_queries.dtype == raw_keys.dtype == raw_values.dtype == torch.bfloat16:
        return False
    if core.rotary_pairs % 8 or 2 * core.rotary_pairs > d:
        return False
    if not (_gain_readable(core.query_weight, d) and _gain_readable(core.key_weight, d)):
        return False
    return _cache_writable(cache, length, core.kv_heads, d)


def mask_served(mask, length: int, rows: int) -> bool:
    """No mask, a string ("causal", or another, which the Core chain ignores) or a boolean
    one of a row per query."""
    if mask is None or isinstance(mask, str):
        return True
    return (mask.dtype == torch.bool and tuple(mask.shape) in ((length, rows), (1, length, rows), (1, 1, length, rows))
            and (rows <= 1 or mask.stride(-1) == 1) and (length <= 1 or mask.stride(-2) >= rows)
            and plain_call(mask))


def _readable_rows(raw: torch.Tensor) -> torch.Tensor:
    """The rows [1, T, width], copied where the kernel could not read them in place."""
    stride = raw.stride(1)
    if (raw.stride(2) != 1 or (raw.shape[1] > 1 and (stride % 8 or stride < raw.shape[2]))
            or raw.data_ptr() % 16):
        raw = raw.clone(memory_format=torch.contiguous_format)
    return raw


def _angle_rows(core, length: int, device):
    """The (cos, sin) rows of this call's positions, or None where the kernel cannot read
    them in place (a table too short among them) or autograd follows them."""
    offset, pairs = core.cache.offset, core.rotary_pairs
    if type(core.angles) is AngleTable:
        cos, sin = core.angles.cos[offset : offset + length], core.angles.sin[offset : offset + length]
    elif type(core.angles) is AngleAtlas:
        rows = core.angles(offset, length)
        cos, sin = rows[:, :pairs], rows[:, pairs : 2 * pairs]
    else:
        cos, sin = core._angles(offset, length, device)
    shape, followed = (length, pairs), torch.is_grad_enabled()
    for rows in (cos, sin):
        if type(rows) not in _PLAIN or (followed and rows.requires_grad):
            return None
        if (rows.dtype != torch.float32 or rows.device != device or rows.shape != shape
                or rows.stride(-1) != 1 or rows.data_ptr() % 16):
            return None
    if length > 1 and (cos.stride(0) % 4 or sin.stride(0) != cos.stride(0)):
        return None
    return cos, sin


def project(core, raw_queries, raw_keys, raw_values):
    """(queries [heads, T, D], keys, values) as `core.project` gives them, the cache written
    and advanced; None, with nothing written, where the angle rows are not for the kernel."""
    length, device = raw_queries.shape[1], raw_queries.device
    angles = None
    if core.rotary_pairs:
        angles = _angle_rows(core, length, device)
        if angles is None:
            return None
    cache = core.cache
    cache.claim(length, core.kv_heads, core.head_dim, raw_keys)
    queries = ops.attention_project(
        _readable_rows(raw_queries), _readable_rows(raw_keys), _readable_rows(raw_values),
        core.query_weight, core.key_weight, angles, cache.keys, cache.values, cache.offset,
        heads=core.heads, kv_heads=core.kv_heads, head_dim=core.head_dim, eps=core.eps, mscale=core.mscale)
    cache.advance(length)
    rows = cache.offset
    return queries, cache.keys[:, :, :rows], cache.values[:, :, :rows]


def prefill(core, raw_queries, raw_keys, raw_values, mask):
    """The context [1, heads, T, D] of a prefill, or None, with nothing written, for a call
    that `core` has to run."""
    if not project_served(core, raw_queries, raw_keys, raw_values):
        return None
    if not 0 < core.scale < math.inf:
        return None
    length = raw_queries.shape[1]
    rows = core.cache.offset + length
    if rows >= MAX_ROWS or not mask_served(mask, length, rows):
        return None
    sinks = core.sinks
    if sinks is not None and (sinks.dtype != torch.bfloat16 or not sinks.is_contiguous()
                              or sinks.numel() != core.heads):
        return None
    projected = project(core, raw_queries, raw_keys, raw_values)
    if projected is None:
        return None
    queries, keys, values = projected
    band = None
    if mask is not None and not isinstance(mask, str):
        band = mask.reshape(mask.shape[-2:])
    out = ops.attention_prefill(queries, keys, values, scale=core.scale,
                                causal=isinstance(mask, str) and mask == "causal", mask=band, sinks=sinks)
    return out.unsqueeze(0)
