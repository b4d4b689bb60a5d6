"""Head dimension 256: dq from the dS that the dk/dv pass hands over (as flex_attention's backward takes it) against the
dq of the recomputing pass, at the edges of the tiles and for grouped heads, masks and a compiled-loop score.  The two
round the same dS to bf16 and sum it in another order: their difference is bounded by one bf16 rounding of the result,
and both are held to the oracle."""
import math

import pytest
import torch

from helpers import assert_close, same_residual_grads
from oracle import mha_oracle as O
from test_gpu_ragged import surrounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk", [(1, 1, 1, 128, 128), (2, 2, 1, 129, 257), (1, 4, 2, 640, 640), (1, 2, 2, 255, 1025)])
@pytest.mark.parametrize("kind", ["none", "causal", "softcap", "alibi"])
def test_dq_from_ds_at_head_dimension_256(kind, B, Hq, Hkv, Sq, Sk):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks, scores
    D, sc = 256, 1 / 16
    mf, sfn, okw = (None, None), None, {}
    if kind == "causal":
        mf, okw = masks.make_causal_mask_fns(128, 128), dict(causal=True)
    elif kind == "softcap":
        sfn, okw = scores.make_softcap_score_fn(5.0), dict(score_mod=O.score_mod_softcap(5.0))
    elif kind == "alibi":
        sfn, okw = scores.make_alibi_global_score_fn(Hq), dict(score_mod=O.score_mod_alibi_global(O.alibi_slopes(Hq)))
    q, k, v, do = O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=torch.bfloat16, seed=Sq)
    qg, kg, vg, dog = [surrounded(x) for x in (q, k, v, do)]
    o, l, m = F._flex_attention_impl(qg, kg, vg, None, None, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], sfn)
    d = F.compute_delta(o, dog)
    kw = dict(block_q=128, block_k_major=128, block_k=128, sm_scale=sc, debug=False, score_fn=sfn, mask_fn=mf[0], block_mask_fn=mf[1])
    dk, dv, ds = F.flash_attention_bwd_dkv(kg, vg, qg, None, None, l, m, d, dog, block_b=1, block_q_major=128, causal=False,
                                           return_ds=True, _wide_ds=True, **kw)
    assert ds is not None
    dq = F.flex_attention_bwd_dq(qg, kg, vg, None, None, l, m, o, dog, d, block_b=1, ds=ds, **kw)
    dk2, dv2 = F.flash_attention_bwd_dkv(kg, vg, qg, None, None, l, m, d, dog, block_b=1, block_q_major=128, causal=False, **kw)
    assert torch.equal(dk, dk2) and torch.equal(dv, dv2)
    same = same_residual_grads(q, k, v, do, o, l, m, sm_scale=sc, **okw)
    assert_close("dq", dq, same[0], torch.bfloat16)   # (dk, dv: the bits of the call without export)
    dq2 = F.flex_attention_bwd_dq(qg, kg, vg, None, None, l, m, o, dog, d, block_b=1, **kw)
    # (both round fp32 sums of the same bf16 products: half a bf16 step of the value each, 2^-8 of it, and where the sum
    # cancels the fp32 orders' difference, far below 1e-5 of its largest terms)
    assert bool(((dq.float() - dq2.float()).abs() <= 2.0 ** -7 * dq2.float().abs() + 1e-3 * float(dq2.float().abs().max())).all())
