"""The prepared calls' autograd function in C++ against the Python one that every other call takes: the same kernels on the same
arguments, so the same bits, for each set of wanted gradients, under the hooks and modes that watch an autograd function, and where
the call is handed to the Python one; where the forward's lists are cut (flexattn_fwd_work), against that forward and its backward."""
import math
import threading

import pytest
import torch

from helpers import assert_close, same_residual_grads
from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu


def agree(got, want):
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def inputs(B=2, Hq=4, Hkv=2, Sq=300, Sk=300, D=128, dtype=torch.bfloat16, seed=0):
    return [t.cuda() for t in O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=dtype, seed=seed)]


def masks_of(causal):
    from flex_attention_tpu_amd import masks
    return masks.make_causal_mask_fns(128, 128) if causal else None


def python_path(q, k, v, pair, sc, causal=False):
    import sys
    fa = sys.modules["flex_attention_tpu_amd.flex_attention"]
    mf, bf = pair or (None, None)
    return fa._FlexAttention.apply(q, k, v, None, (None, mf, bf, None, causal, sc, 128, 128))


def taken(q, k, v, pair, sc, **kw):
    """flex_attention's result, and whether the C++ function made it."""
    import flex_attention_tpu_amd as F
    o = F.flex_attention(q, k, v, None, pair, sm_scale=sc, **kw)
    return o, o.grad_fn is not None and "_FlexAttentionBackward" not in type(o.grad_fn).__name__


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.bfloat16, 64), (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize("Sq,Sk,causal", [(128, 128, False), (300, 300, True), (257, 640, False)])
@pytest.mark.parametrize("wanted", ["qkv", "q", "k", "v", "kv"])
def test_same_bits_as_the_python_function(wanted, Sq, Sk, causal, dtype, D):
    q, k, v, do = inputs(Sq=Sq, Sk=Sk, D=D, dtype=dtype)
    sc, pair = 1 / math.sqrt(D), masks_of(causal)
    leaves = [t for n, t in zip("qkv", (q, k, v)) if n in wanted]
    for t in leaves:
        t.requires_grad_(True)
    o, native = taken(q, k, v, pair, sc)
    assert native
    want = python_path(q, k, v, pair, sc)
    with torch.no_grad():
        assert torch.equal(taken(q, k, v, pair, sc)[0], o)
    agree((o, *torch.autograd.grad(o, leaves, do)), (want, *torch.autograd.grad(want, leaves, do)))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal", [(1, 2, 1, 1024, 1024, True), (1, 2, 2, 1100, 1100, True), (2, 1, 1, 200, 1601, False)])
def test_cut_lists(B, Hq, Hkv, Sq, Sk, causal):
    """Small grids of long lists: the C++ forward brings the memory for the parts' sums, and its backward takes the residuals of
    the merged rows."""
    from flex_attention_tpu_amd import _lib, _plans
    from flex_attention_tpu_amd.block_mask import spec_of
    q, k, v, do = inputs(B, Hq, Hkv, Sq, Sk)
    sc, pair = 1 / math.sqrt(128), masks_of(causal)
    spec = spec_of(*(pair or (None, None)))
    o, l, m = _plans.forward(q, k, v, spec, sc, True, with_work=True)
    assert next(p for p in reversed(_plans._plans._d.values())).work_bytes >= 2 * q.numel() * 4   # (two parts or more)
    whole, _, _ = _plans.forward(q, k, v, spec, sc, True)
    assert not torch.equal(o, whole)
    want = (o, *_plans.backward(q, k, v, l, m, o, do, spec, sc))
    with torch.no_grad():
        assert torch.equal(taken(q, k, v, pair, sc)[0], o)
    for t in (q, k, v):
        t.requires_grad_(True)
    for _ in range(2):
        got, native = taken(q, k, v, pair, sc)
        assert native
        agree((got, *torch.autograd.grad(got, (q, k, v), do)), want)
    cpu = [t.detach().cpu() for t in (q, k, v, do)]
    assert_close("o", o, O.mha_reference(*cpu[:3], sm_scale=sc, causal=causal), torch.bfloat16)
    for name, t, r in zip(("dq", "dk", "dv"), want[1:], same_residual_grads(*cpu, o, l, m, sm_scale=sc, causal=causal)):
        assert_close(name, t, r, torch.bfloat16)


def test_views_hooks_and_repeated_backward():
    sc, pair = 1 / math.sqrt(128), masks_of(True)
    q, k, v, do = inputs()
    for t in (q, k, v):
        t.requires_grad_(True)
    want = torch.autograd.grad(taken(q, k, v, pair, sc)[0], (q, k, v), do)
    agree(want, torch.autograd.grad(python_path(q, k, v, pair, sc), (q, k, v), do))

    def check(o, do=do, **kw):
        got = torch.autograd.grad(o, (q, k, v), do, **kw)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    o, native = taken(q, k, v, pair, sc)
    assert native
    check(o, retain_graph=True)
    check(o, do=do.transpose(1, 2).contiguous().transpose(1, 2))   # (a gradient of other strides; frees the graph)
    with pytest.raises(RuntimeError, match="backward through the graph a second time"):
        torch.autograd.grad(o, (q, k, v), do)
    with torch.autograd.graph.save_on_cpu():
        o, native = taken(q, k, v, pair, sc)
    assert native
    check(o)
    o = torch.utils.checkpoint.checkpoint(lambda *a: taken(*a, pair, sc)[0], q, k, v, use_reentrant=False)
    check(o)
    # operands at an address that is no multiple of 16 bytes
    off = [torch.cat([t.detach().new_zeros(1), t.detach().flatten()])[1:].view(t.shape).requires_grad_(True) for t in (q, k, v)]
    o, native = taken(*off, pair, sc)
    assert native and all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, off, do), want))
    # an operand that changes before the backward
    x = q.detach().clone().requires_grad_(True)
    y = x * 1.0
    o, _ = taken(y, k, v, pair, sc)
    with torch.no_grad():
        y.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(o, x, do)


def test_calls_that_stay_with_the_python_function():
    import flex_attention_tpu_amd as F
    sc = 1 / math.sqrt(128)
    q, k, v, do = inputs()
    q.requires_grad_(True)
    strided = q.detach().transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(True)
    o, native = taken(strided, k, v, None, sc)
    assert not native
    agree((taken(q, k, v, None, sc)[0],), (o,))
    with torch.autograd.forward_ad.dual_level():
        assert not taken(q, k, v, None, sc)[1]
    for bad in ((q[0], k, v), (q, k[:, :, :-1], v), (q, k.float(), v), (q, k, v.cpu()), (q[:, :3].contiguous(), k, v)):
        for call in (lambda: F.flex_attention(*bad, sm_scale=sc), lambda: python_path(*bad, None, sc)):
            with pytest.raises(ValueError):
                call()
    for scale in (0.0, -1.0, math.inf, math.nan):   # (refused by the library, behind the C++ function)
        with pytest.raises(ValueError, match="sm_scale"):
            F.flex_attention(q, k, v, sm_scale=scale)


@pytest.mark.parametrize("D,S,mask", [(128, 512, "causal"), (64, 300, "causal"), (128, 384, "window"), (256, 512, "causal"), (128, 512, "documents")])
def test_under_compilation(D, S, mask):
    """torch.compile makes the call between its graphs: its first call of a combination as well as later ones, with the same bits."""
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import block_mask, masks
    pair = {"causal": lambda: masks_of(True), "window": lambda: masks.make_causal_sliding_window_mask_fns(128, 128, 100),
            "documents": lambda: masks.make_jagged_mask_fns(128, 128, [200, S - 200])}[mask]()
    q, k, v, do = inputs(Sq=S, Sk=S, D=D)
    for t in (q, k, v):
        t.requires_grad_(True)
    block_mask._map_cache.clear()
    torch._dynamo.reset()
    f = torch.compile(lambda q, k, v: 2 * F.flex_attention(q * 1, k, v, None, pair) + 0, backend="eager")
    got = [torch.autograd.grad(f(q, k, v), (q, k, v), do) for _ in range(2)]
    o = 2 * F.flex_attention(q * 1, k, v, None, pair) + 0
    want = torch.autograd.grad(o, (q, k, v), do)
    assert torch.equal(f(q, k, v), o)
    for g in got:
        agree(g, want)


def test_streams_and_threads():
    sc, pair = 1 / math.sqrt(128), masks_of(True)
    want, errors = {}, []
    sets = [inputs(seed=s) for s in range(4)]
    for n, (q, k, v, do) in enumerate(sets):
        for t in (q, k, v):
            t.requires_grad_(True)
        want[n] = torch.autograd.grad(taken(q, k, v, pair, sc)[0], (q, k, v), do)
    torch.cuda.synchronize()

    def work(n):
        try:
            q, k, v, do = sets[n]
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(10):
                    o, native = taken(q, k, v, pair, sc)
                    got = torch.autograd.grad(o, (q, k, v), do)
                    assert native
            stream.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want[n]))
        except BaseException as e:
            errors.append(e)
    threads = [threading.Thread(target=work, args=(n,)) for n in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_captured_and_replayed():
    from flex_attention_tpu_amd import _plans, block_mask
    sc, pair = 1 / math.sqrt(64), masks_of(True)
    q, k, v, do = inputs(Sq=384, Sk=384, D=64, dtype=torch.float32)
    for t in (q, k, v):
        t.requires_grad_(True)

    def step():
        o, native = taken(q, k, v, pair, sc)
        assert native
        return (o, *torch.autograd.grad(o, (q, k, v), do))
    step()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    block_mask._map_cache.clear()   # (the captured call builds its maps, which the graph's memory then holds)
    _plans._attend_plans.clear()
    with torch.cuda.graph(graph, stream=side):
        got = step()
    assert all(torch.isfinite(t).all() for t in step())   # (a call between capture and replay: it builds maps of its own)
    block_mask._map_cache.clear()
    for seed in (1, 2, 3):
        for t, n in zip((q, k, v, do), inputs(Sq=384, Sk=384, D=64, dtype=torch.float32, seed=seed)):
            t.data.copy_(n)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, step()):
            assert torch.equal(a, b)


@pytest.mark.parametrize("known", [False, True])
def test_a_captured_call_keeps_its_maps(known):
    """The graph holds the maps' addresses: they live as long as the graph, whatever the caches drop, and a map that only a replay
    builds serves no call outside."""
    import gc
    import weakref

    from flex_attention_tpu_amd import _plans, block_mask
    sc, pair = 1 / math.sqrt(64), masks_of(True)
    q, k, v, do = inputs(Sq=640, Sk=640, D=64)
    q.requires_grad_(True)
    S = 640 if known else 384   # (the kernels loaded; the maps of 640 known or not)
    warm = [t.detach()[:, :, :S].contiguous().requires_grad_(n == 0) for n, t in enumerate((q, k, v))]
    torch.autograd.grad(taken(*warm, pair, sc)[0], warm[0], do[:, :, :S].contiguous())
    if not known:
        block_mask._map_cache.clear()
        _plans._attend_plans.clear()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    gc.collect()
    before = set(block_mask._captures)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        o, _ = taken(q, k, v, pair, sc)
        dq, = torch.autograd.grad(o, q, do)
    capture, = set(block_mask._captures) - before
    maps = list(block_mask._captures[capture].things.values())
    used = [weakref.ref(m) for m in maps]
    assert used and all(m.captured is not known and any(m is c for c in block_mask._map_cache._d.values()) is known for m in maps)
    del maps
    o1, _ = taken(q, k, v, pair, sc)   # (in front of the first replay: on maps of its own)
    dq1, = torch.autograd.grad(o1, q, do)
    block_mask._map_cache.clear()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, o1) and torch.equal(dq, dq1)
        block_mask.release_ended()
        gc.collect()
        assert all(r() is not None for r in used)
    o2, _ = taken(q, k, v, pair, sc)
    assert torch.equal(o, o2) and torch.equal(dq, torch.autograd.grad(o2, q, do)[0])
    block_mask._map_cache.clear()
    del graph
    gc.collect()
    block_mask.release_ended()
    assert capture not in block_mask._captures and all(r() is None for r in used)


def test_a_captured_call_keeps_its_ids_and_slopes():
    """The caches of document ids and position-bias slopes drop the arrays that a captured call reads, and their memory goes to other
    tensors: the replays still read them."""
    import gc

    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _common, block_mask, masks, scores
    pair, sfn, sc = masks.make_jagged_mask_fns(128, 128, [150, 250, 112]), scores.make_alibi_global_score_fn(4), 1 / math.sqrt(128)
    q, k, v, do = inputs(Sq=512, Sk=512)
    q.requires_grad_(True)

    def step():
        o = F.flex_attention(q, k, v, sfn, pair, sm_scale=sc)
        return o.detach(), torch.autograd.grad(o, q, do)[0]
    want = step()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = step()
    for cache in (block_mask._map_cache, block_mask._doc_cache, block_mask._range_cache, _common._slopes_cache):
        cache.clear()
    gc.collect()
    others = [torch.full((n,), -1, dtype=torch.int32, device="cuda") for n in (4, 16, 64, 256, 512, 1024) for _ in range(64)]
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(int(t.max()) == -1 for t in others)


def test_names_of_captures():
    """One name per capture, the same on its forked streams; told as ended when the graph has been dropped or reset, not before."""
    import ctypes as C
    import gc

    from flex_attention_tpu_amd import _lib, block_mask
    lib, x = _lib.load(), torch.zeros(8, device="cuda")

    def name():
        return lib.flexattn_capture_token(torch.cuda.current_stream().cuda_stream)

    def ended():
        out = (C.c_int64 * 4)()
        return sorted(out[:lib.flexattn_captures_ended(out, 4)])
    gc.collect()
    block_mask.release_ended()
    side, fork = torch.cuda.Stream(), torch.cuda.Stream()
    assert name() == 0
    with torch.cuda.stream(side):
        assert name() == 0
    graphs, names = [], []
    for _ in range(3):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=side):
            names.append(name())
            x.add_(1)
            fork.wait_stream(side)
            with torch.cuda.stream(fork):
                assert name() == names[-1]
                x.add_(1)
            side.wait_stream(fork)
            assert name() == names[-1]
        graphs[-1].replay()
        torch.cuda.synchronize()
    assert len(set(names)) == 3 and min(names) > 0 and ended() == [] and x[0] == 6
    graphs[1].reset()
    assert ended() == [names[1]]
    graphs[0].replay()
    torch.cuda.synchronize()
    assert ended() == [] and x[0] == 8
    del graphs
    gc.collect()
    assert ended() == sorted((names[0], names[2]))
