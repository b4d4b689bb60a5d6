"""Prepared launches (_plans.py) against the general path of the entry points: the same bits, for every mask that takes
them, dtypes, grouped heads, ragged lengths, a second stream, and threads that use one combination at once."""
import math
import threading

import pytest
import torch

from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.bfloat16, 64), (torch.bfloat16, 256), (torch.float32, 64)])
@pytest.mark.parametrize("mask", ["none", "causal", "window", "s2", "flag"])
def test_prepared_calls_give_the_general_path_s_bits(mask, dtype, D, monkeypatch):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _plans, masks
    pair = {"none": None, "flag": None, "causal": masks.make_causal_mask_fns(128, 128),
            "window": masks.make_causal_sliding_window_mask_fns(128, 128, 200), "s2": masks.make_s2_mask_fns(128, 128, 64, 32)
            if hasattr(masks, "make_s2_mask_fns") else masks.make_causal_mask_fns(128, 128)}[mask]
    for B, Hq, Hkv, S in ((1, 2, 1, 128), (2, 4, 2, 321), (1, 2, 2, 640)):
        q, k, v, do = (x.cuda() for x in O.make_inputs(B, Hq, Hkv, S, S, D, dtype=dtype, seed=S))
        for t in (q, k, v):
            t.requires_grad_(True)

        def call():
            o = F.flex_attention(q, k, v, None, pair, causal=mask == "flag", sm_scale=0.9 / math.sqrt(D))
            return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))
        got = [call(), call()]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            got.append(call())
        torch.cuda.current_stream().wait_stream(side)
        threads, results = [], [None] * 3
        for i in range(3):
            def work(i=i):
                with torch.cuda.stream(torch.cuda.Stream()):
                    results[i] = call()
                    torch.cuda.current_stream().synchronize()
            torch.cuda.synchronize()
            threads.append(threading.Thread(target=work))
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        with monkeypatch.context() as mp:
            mp.setattr(_plans, "takes", lambda *a: False)
            want = call()
        for g in got + results:
            assert all(torch.equal(a, b) for a, b in zip(g, want)), (mask, S)
    assert len(_plans._plans) <= _plans._plans.maxsize


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.bfloat16, 64), (torch.bfloat16, 256), (torch.float32, 64)])
@pytest.mark.parametrize("mask", ["none", "causal", "window", "s2"])
def test_the_prepared_passes_are_the_ones_that_run(mask, dtype, D, monkeypatch):
    """The entry points themselves, forward and backward (flex_attention's own backward hands dS over for some of these
    combinations and takes the prepared one for the others): prepared passes are taken once each, or, switched off, not at
    all, and give the same bits."""
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _plans, masks
    from flex_attention_tpu_amd.flex_attention import flex_attention_bwd
    mf, bf = {"none": (None, None), "causal": masks.make_causal_mask_fns(128, 128),
              "window": masks.make_causal_sliding_window_mask_fns(128, 128, 200), "s2": masks.make_s2_mask_fns(128, 128, 64, 32)}[mask]
    taken = []
    for name in ("forward", "backward"):
        real = getattr(_plans, name)
        monkeypatch.setattr(_plans, name, lambda *a, real=real, name=name: taken.append(name) or real(*a))
    for B, Hq, Hkv, S in ((1, 2, 1, 128), (2, 4, 2, 321)):
        q, k, v, do = (x.cuda() for x in O.make_inputs(B, Hq, Hkv, S, S, D, dtype=dtype, seed=S))
        sc = 0.9 / math.sqrt(D)

        def call():
            o, l, m = F._flex_attention_impl(q, k, v, None, None, True, False, sc, 1, 128, 128, 128, False, bf, mf, None)
            return (o, l, m, *flex_attention_bwd(q, k, v, None, None, l, m, o, do, block_q=128, block_k=128, sm_scale=sc, mask_fn=mf, block_mask_fn=bf))
        got = call()
        assert taken == ["forward", "backward"]
        with monkeypatch.context() as mp:
            mp.setattr(_plans, "takes", lambda *a: False)
            want = call()
        assert taken == ["forward", "backward"]
        taken.clear()
        assert all(torch.equal(a, b) for a, b in zip(got, want)), S


def test_plans_pin_no_block_maps():
    """A map that its cache has dropped is gone although a plan points at it; the plan is made again, with the same bits."""
    import gc
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _plans, block_mask, masks
    pair = masks.make_causal_mask_fns(128, 128)
    q, k, v, do = (x.cuda().requires_grad_(True) for x in O.make_inputs(1, 2, 2, 384, 384, 128, dtype=torch.bfloat16, seed=4))

    def call():
        o = F.flex_attention(q, k, v, None, pair)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))
    want = call()
    torch.cuda.synchronize()
    plans = list(_plans._plans._d.values())
    block_mask._map_cache.clear()
    gc.collect()
    assert plans and all(ref() is None for p in plans for ref in p.maps)
    assert all(torch.equal(a, b) for a, b in zip(call(), want))
    assert len(_plans._plans) <= _plans._plans.maxsize
