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
