"""bf16 head dimensions up to 64 on the streams of head dimension 64: masks, grouped heads, ragged lengths, several
work items per work-group, and a scale that folds into Q in no kernel but the backward's own variant; NaN around every
operand.  Tolerances: helpers.assert_close."""
import math
import types

import pytest
import torch

from helpers import assert_close, same_residual_grads
from oracle import mha_oracle as O
from test_gpu_ragged import surrounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D", [(2, 4, 2, 128, 128, 64), (1, 2, 2, 513, 777, 64), (1, 6, 2, 1000, 1000, 40),
                                              (2, 2, 1, 640, 2048, 64), (4, 16, 16, 1024, 1024, 64)])
@pytest.mark.parametrize("mask", ["none", "causal", "window", "documents", "unsorted"])
def test_head_dim_64(mask, B, Hq, Hkv, Sq, Sk, D):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks
    sc = 1 / math.sqrt(D)
    mf, sid, okw = (None, None), None, {}
    if mask == "causal":
        mf, okw = masks.make_causal_mask_fns(128, 128), dict(causal=True)
    elif mask == "window":
        W = 150 + max(0, Sq - Sk)      # (every query keeps a key)
        mf, okw = masks.make_sliding_window_mask_fns(128, 128, W), dict(window_size=W)
    elif mask != "none":
        ids_q, ids_k = (torch.arange(S) * 3 // S for S in (Sq, Sk))
        if mask == "unsorted":
            ids_k = ids_k.flip(0)
        sid, okw = types.SimpleNamespace(q=ids_q, kv=ids_k), dict(mask=ids_q[:, None] == ids_k[None, :])
    q, k, v, do = O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=torch.bfloat16, seed=Sq + D)
    ro, rl, rm = O.mha_reference(q, k, v, sm_scale=sc, save_residuals=True, **okw)
    qg, kg, vg, dog = [surrounded(x) for x in (q, k, v, do)]
    o, l, m = F._flex_attention_impl(qg, kg, vg, None, sid, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], None)
    assert_close("o", o, ro, torch.bfloat16)
    assert_close("lse", m + l.log(), rm + rl.log(), torch.bfloat16)
    l, m, os_ = surrounded(l), surrounded(m), surrounded(o)
    d = surrounded(F.compute_delta(os_, dog))
    kw = dict(block_q=128, block_k_major=128, block_k=128, debug=False, score_fn=None, mask_fn=mf[0], block_mask_fn=mf[1])
    dq = F.flex_attention_bwd_dq(qg, kg, vg, None, sid, l, m, os_, dog, d, block_b=1, sm_scale=sc, **kw)
    dk, dv = F.flash_attention_bwd_dkv(kg, vg, qg, None, sid, l, m, d, dog, block_b=1, block_q_major=128, causal=False, sm_scale=sc, **kw)
    same = same_residual_grads(q, k, v, do, o, l, m, sm_scale=sc, **okw)
    for name, t, r in zip(("dq", "dk", "dv"), (dq, dk, dv), same):
        assert_close(name, t, r, torch.bfloat16)


def test_exact_scale_dq_stream_is_reached():
    """The dq stream that scales the fp32 product: the C call takes any scale (the Python entry points hand head
    dimension 64 to it only with scales that fold, so it is called here directly), against the zero-padded kernels."""
    import ctypes as C
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _lib
    from flex_attention_tpu_amd._common import kernel_block_map, stream_of
    from flex_attention_tpu_amd.flex_attention_dq_bwd import bwd_params
    from flex_attention_tpu_amd.masks import MaskSpec
    B, H, S, D, sc = 1, 2, 384, 64, 0.7
    q, k, v, do = (x.cuda() for x in O.make_inputs(B, H, H, S, S, D, dtype=torch.bfloat16, seed=5))
    o, l, m = F._flex_attention_impl(q, k, v, None, None, True, False, sc, 1, 128, 128, 128, False, None, None, None)
    d = F.compute_delta(o, do)
    dq = torch.empty_like(q)
    bm = kernel_block_map(_lib.PASS_DQ, MaskSpec(), q, S, S, D)
    p = bwd_params(q, k, v, l, m, do, d, sc, None, MaskSpec(), bm, 1, 1, dq=dq)
    _lib.check(_lib.load().flexattn_bwd_dq(C.byref(p), stream_of(q)))
    same = same_residual_grads(*(x.cpu() for x in (q, k, v, do)), o, l, m, sm_scale=sc)
    assert_close("dq", dq, same[0], torch.bfloat16, tensor_scale=True)


@pytest.mark.parametrize("D", [8, 16, 24])
@pytest.mark.parametrize("mask", ["none", "causal"])
def test_scales_that_do_not_fold(mask, D):
    """1 / sqrt(D) of the smallest head dimensions is a scale that the kernels of 128 columns do not fold into bf16 Q: o, l
    and m are theirs, and the backward (at 64 columns, dq by the stream that scales the fp32 product) gives what they
    give on zero-padded operands."""
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks
    mf = masks.make_causal_mask_fns(128, 128) if mask == "causal" else (None, None)
    B, H, S, sc = 2, 2, 321, 1 / math.sqrt(D)
    ts = O.make_inputs(B, H, H, S, S, D, dtype=torch.bfloat16, seed=D)

    def passes(q, k, v, do):
        o, l, m = F._flex_attention_impl(q, k, v, None, None, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], None)
        kw = dict(block_b=1, block_q=128, block_k_major=128, block_k=128, sm_scale=sc, debug=False, mask_fn=mf[0], block_mask_fn=mf[1])
        dq, d = F.flex_attention_bwd_dq(q, k, v, None, None, l, m, o, do, None, return_delta=True, **kw)
        return (o, l, m, dq, *F.flash_attention_bwd_dkv(k, v, q, None, None, l, m, d, do, block_q_major=128, causal=False, **kw))
    got = passes(*(x.cuda() for x in ts))
    want = passes(*(torch.nn.functional.pad(x, (0, 128 - D)).cuda() for x in ts))
    for name, a, b in zip(("o", "l", "m", "dq", "dk", "dv"), got, want):
        assert torch.equal(a, b[..., :D] if b.ndim == 4 else b), name
    same = same_residual_grads(*ts, *got[:3], sm_scale=sc, **(dict(causal=True) if mask == "causal" else {}))
    for name, t, r in zip(("dq", "dk", "dv"), got[3:], same):
        assert_close(name, t, r, torch.bfloat16)
