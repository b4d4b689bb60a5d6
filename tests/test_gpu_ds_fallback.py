"""The backward that hands dS from the dk/dv to the dq pass, where there is no room for the buffer, or not beside what else
the backward needs, or where its index cannot be built: it falls back to the recomputing passes and returns what those
return, bit for bit."""
import math
import sys

import pytest
import torch

from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu


def step(kind, S=321):
    """(call, recompute): one forward and backward, and the gradients of the recomputing passes on its residuals."""
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import scores
    B, H, D = 2, 2, 256 if kind == "d256" else 128
    sc = 1 / math.sqrt(D)
    sfn = scores.make_softcap_score_fn(5.0) if kind == "softcap" else None
    q, k, v, do = (x.cuda() for x in O.make_inputs(B, H, H, S, S, D, dtype=torch.bfloat16, seed=S))
    ab = torch.randn(1, H, S, S, generator=torch.Generator().manual_seed(1)).cuda().requires_grad_(True) if kind == "bias" else None
    leaves = [t.requires_grad_(True) for t in (q, k, v)] + ([ab] if ab is not None else [])

    def call():
        o = F.flex_attention(q, k, v, sfn, None, sm_scale=sc, ab=ab)
        return torch.autograd.grad(o, leaves, do)

    def recompute():
        with torch.no_grad():
            o, l, m = F._flex_attention_impl(q, k, v, ab, None, True, False, sc, 1, 128, 128, 128, False, None, None, sfn)
            kw = dict(block_b=1, block_q=128, block_k_major=128, block_k=128, sm_scale=sc, debug=False, score_fn=sfn)
            d = F.compute_delta(o, do)
            dq = F.flex_attention_bwd_dq(q, k, v, ab, None, l, m, o, do, d, return_dab=ab is not None, **kw)
            dk, dv = F.flash_attention_bwd_dkv(k, v, q, ab, None, l, m, d, do, block_q_major=128, causal=False, **kw)
            return (dq[0], dk, dv, dq[1]) if ab is not None else (dq, dk, dv)
    return call, recompute


def same(a, b):
    return len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("kind", ["d256", "bias", "softcap"])
def test_no_room_for_ds(kind, monkeypatch):
    from flex_attention_tpu_amd import flex_attention_dkv_kernel as dkv
    call, recompute = step(kind)
    asked = []
    monkeypatch.setattr(dkv, "alloc_ds", lambda *a: asked.append(a) or None)
    assert same(call(), recompute()) and len(asked) == 1


@pytest.mark.parametrize("kind", ["d256", "bias", "softcap"])
def test_no_room_beside_ds(kind, monkeypatch):
    """Every allocation behind the buffer's fails while the buffer lives."""
    fa = sys.modules["flex_attention_tpu_amd.flex_attention"]   # (the package exports the function under the same name)
    call, recompute = step(kind)
    real, seen = fa.flex_attention_bwd_dq, []

    def dq_pass(*a, ds=None, **kw):
        seen.append(ds is not None)
        if ds is not None:
            raise torch.cuda.OutOfMemoryError("no room beside dS")
        return real(*a, **kw)
    monkeypatch.setattr(fa, "flex_attention_bwd_dq", dq_pass)
    assert same(call(), recompute()) and seen[0]


def test_the_bias_gradient_is_allocated_before_ds(monkeypatch):
    """Needed with and without the hand-over: were dS allocated first, the bias gradient could fail beside it."""
    from flex_attention_tpu_amd import flex_attention_dkv_kernel as dkv
    call, _ = step("bias")
    order, ds, dab = [], dkv.alloc_ds, dkv.alloc_dab
    monkeypatch.setattr(dkv, "alloc_ds", lambda *a: order.append("ds") or ds(*a))
    monkeypatch.setattr(dkv, "alloc_dab", lambda *a: order.append("dab") or dab(*a))
    call()
    assert order == ["dab", "ds"]


@pytest.mark.parametrize("kind", ["d256", "bias", "softcap"])
def test_captured_without_a_call_before(kind):
    """A capture of a shape that no call has had (the kernels themselves loaded by another shape): the number of tile pairs
    would have to come back to the host, so the captured backward recomputes."""
    from flex_attention_tpu_amd import _plans, block_mask
    step(kind)[0]()
    step(kind)[1]()
    call, recompute = step(kind, S=467)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = call()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        block_mask._map_cache.clear()   # (the captured call's map lives in the graph)
        _plans._plans.clear()
        assert same(got, recompute())
