"""The router's product path (csrc/router.hip, router_logits_kernel): more rows than the decode
path's with the logits written. Every logit has to be the correctly rounded bf16 of the exact
dot product of the normalized row and the expert's row, whatever its error bound leaves to
recompute, so it is compared bit for bit with the float64 product rounded once.

Rows straddle a 16-token tile and both ways of splitting a workgroup; the values are plain
ones, ones with outlying columns (a sum far larger than the logit), norm weights and gates
near the ends of bf16's range, and rows and experts that are zero or not finite.
"""

import numpy as np
import pytest
import torch

from mlx_omnia_amd.kernels.leaf import RMSNormLeaf
from mlx_omnia_amd.kernels.route import ResidualRouter, Routing
from mlx_omnia_amd.runtime import ops
from oracle.activations import f64_to_bf16
from oracle.bf16 import from_float, to_f32
from util import bits_of, to_device

pytestmark = pytest.mark.gpu


def _inputs(rows, hidden, experts, kind, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, hidden), dtype=np.float32)
    r = rng.standard_normal((rows, hidden), dtype=np.float32)
    w = 1.0 + 0.1 * rng.standard_normal(hidden)
    gate = 0.02 * rng.standard_normal((experts, hidden), dtype=np.float32)
    if kind == "outliers":
        x[:, ::97] *= 300.0
        gate[:, ::89] *= 50.0
    elif kind == "small gate":       # subnormal weights and products
        gate *= 2.0 ** -124
        w *= 2.0 ** 20
    elif kind == "large norm":
        w *= 2.0 ** 70
        gate *= 2.0 ** -80
        gate[:, ::5] = 2.0 ** -130
    elif kind == "special":
        x[3], r[3] = 0.0, 0.0
        gate[5] = 0.0
        gate[7, 11] = np.inf
        gate[9, 12] = np.nan
    return from_float(x), from_float(r), from_float(w), from_float(gate)


@pytest.mark.parametrize("rows,hidden,experts", [
    (257, 2048, 128), (1280, 2048, 128),      # the least and the most rows of this shape
    (129, 2048, 256), (1040, 2048, 256),      # one expert tile a workgroup; two
    (257, 4096, 128), (2063, 4096, 128),
    (129, 4096, 256), (1030, 4096, 256),
])
def test_every_logit_is_the_rounded_exact_product(rows, hidden, experts):
    kinds = ["plain", "outliers", "small gate", "large norm", "special"] if rows < 300 else ["plain"]
    for kind in kinds:
        print(f"router product path rows={rows} hidden={hidden} experts={experts} {kind}", flush=True)
        x, r, w, gate = _inputs(rows, hidden, experts, kind, seed=rows + hidden + experts)
        xd, rd, wd, gd = (to_device(v) for v in (x, r, w, gate))
        s, n, logits, idx, wts = ops.residual_rms_router(xd, rd, wd, gd, k=8, eps=1e-6, emit_logits=True)
        s2, n2 = ops.add_rms_norm(xd, rd, wd, 1e-6)
        assert torch.equal(s, s2) and torch.equal(n.view(torch.int16), n2.view(torch.int16))
        with np.errstate(invalid="ignore", over="ignore"):
            exact = to_f32(bits_of(n)).astype(np.float64) @ to_f32(gate).astype(np.float64).T
        got, finite = bits_of(logits), np.isfinite(exact)
        want = f64_to_bf16(np.where(finite, exact, 0.0))
        assert np.array_equal(got[finite] & 0x7FFF == 0, want[finite] & 0x7FFF == 0)
        real = finite & (want & 0x7FFF != 0)
        assert np.array_equal(got[real], want[real])
        widened = to_f32(got)
        assert np.array_equal(np.isnan(widened[~finite]), np.isnan(exact[~finite]))
        assert np.array_equal(np.isposinf(widened), np.isposinf(exact) | (finite & (exact >= 2.0 ** 128)))
        if kind != "special":
            idx2, wts2 = ops.softmax_topk(logits, 8)
            assert torch.equal(idx, idx2) and torch.equal(wts, wts2)
            bias = torch.linspace(-0.1, 0.1, experts, device="cuda")
            _, _, same, keys, _, _ = ops.residual_rms_router_sigmoid(xd, rd, wd, gd, bias, k=8, eps=1e-6)
            assert torch.equal(same, logits)
            assert torch.equal(ops.sigmoid_topk(logits, bias, 8, emit_keys=True, select=False)[2].view(torch.int32),
                               keys.view(torch.int32))


@pytest.mark.parametrize("rows,hidden,experts", [
    (33, 2048, 128), (300, 2048, 256), (33, 4096, 128), (300, 4096, 256),
])
def test_keys_without_the_logits_are_those_of_the_logits(rows, hidden, experts):
    """The fused kernels, every logit exact in them: the same keys and selection as from the
    logits written by the other paths."""
    print(f"router keys alone rows={rows} hidden={hidden} experts={experts}", flush=True)
    xd, rd, wd, gd = (to_device(v) for v in _inputs(rows, hidden, experts, "outliers", seed=rows + experts))
    bias = torch.linspace(-0.1, 0.1, experts, device="cuda")
    want = ops.residual_rms_router_sigmoid(xd, rd, wd, gd, bias, k=8, eps=1e-6, select=True)
    got = ops.residual_rms_router_sigmoid(xd, rd, wd, gd, bias, k=8, eps=1e-6, emit_logits=False, select=True)
    assert got[2] is None
    for ours, theirs in zip(got[:2] + got[3:], want[:2] + want[3:]):
        assert torch.equal(ours.view(torch.int16), theirs.view(torch.int16))


@pytest.mark.parametrize("hidden", [2048, 4096])
@pytest.mark.parametrize("rows", [64, 65, 128, 129])
def test_a_selection_takes_one_dispatch_where_the_host_is_the_bound(monkeypatch, rows, hidden):
    """Eager calls of hidden 2048 above 64 rows, captured ones and hidden 4096 above 128; the
    selection is the same bits either way."""
    print(f"router selection rows={rows} hidden={hidden}", flush=True)
    asked = []
    router_of = ops.residual_rms_router
    monkeypatch.setattr(ops, "residual_rms_router",
                        lambda *args, **kw: asked.append(kw["emit_logits"]) or router_of(*args, **kw))
    xd, rd, wd, gd = (to_device(v) for v in _inputs(rows, hidden, 128, "outliers", seed=rows))
    router = ResidualRouter(RMSNormLeaf(wd, 1e-6), gd, routing=Routing(experts=128, k=8))
    eager = router(xd, rd)
    assert asked == [rows <= (64 if hidden == 2048 else 128)]
    want = router_of(xd, rd, wd, gd, k=8, eps=1e-6, emit_logits=not asked[0])
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = router(xd, rd)
    assert asked[1] == (rows <= 128)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for got in (eager, captured):
            for ours, theirs in zip(got, want[:2] + want[3:]):
                assert torch.equal(ours.view(torch.int16), theirs.view(torch.int16))
