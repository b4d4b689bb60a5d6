"""flex_attention's gradients with a trained bias (the bias gradient out of the dk/dv pass, dq from its dS) at the edges of
the tiles, for every way a bias broadcasts, masks, grouped heads, scores and bias dtypes, against the oracle on the kernels'
own forward.  Tolerances: helpers.assert_close; the bias gradient P (dP - delta) by its values, relative where they
exceed 1, as the dq pass's is in test_gpu_ragged."""
import math

import pytest
import torch

from helpers import assert_close, same_residual_grads
from oracle import mha_oracle as O
from test_gpu_ragged import surrounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D", [(1, 2, 2, 128, 128, 128), (2, 4, 2, 129, 257, 128), (3, 2, 1, 321, 255, 64), (2, 2, 2, 100, 300, 96)])
@pytest.mark.parametrize("ab_shape", ["11", "1h", "b1", "bh"])
@pytest.mark.parametrize("kind", ["plain", "causal", "softcap", "bf16 bias"])
def test_bias_gradient(kind, ab_shape, B, Hq, Hkv, Sq, Sk, D):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks, scores
    sc, pair, sfn, okw = 1 / math.sqrt(D), None, None, {}
    if kind == "causal":
        pair, okw = masks.make_causal_mask_fns(128, 128), dict(causal=True)
    elif kind == "softcap":
        sfn, okw = scores.make_softcap_score_fn(5.0), dict(score_mod=O.score_mod_softcap(5.0))
    ab = torch.randn(B if ab_shape[0] == "b" else 1, Hq if ab_shape[1] == "h" else 1, Sq, Sk, generator=torch.Generator().manual_seed(3))
    if kind == "bf16 bias":
        ab = ab.bfloat16()
    okw["ab"] = ab.float().expand(B, Hq, Sq, Sk)
    q, k, v, do = O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=torch.bfloat16, seed=Sq + D)
    qg, kg, vg, abg = [surrounded(x).requires_grad_(True) for x in (q, k, v, ab)]
    o = F.flex_attention(qg, kg, vg, sfn, pair, sm_scale=sc, ab=abg)
    dq, dk, dv, dab = torch.autograd.grad(o, (qg, kg, vg, abg), surrounded(do))
    mf = pair or (None, None)
    with torch.no_grad():
        o2, l, m = F._flex_attention_impl(qg, kg, vg, abg, None, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], sfn)
    assert torch.equal(o2, o)
    same = same_residual_grads(q, k, v, do, o, l, m, sm_scale=sc, **okw)
    for name, t, r in zip(("dq", "dk", "dv"), (dq, dk, dv), same):
        assert_close(name, t, r, torch.bfloat16)
    ref = O.mha_bwd_reference(q, k, v, o.detach().float().cpu(), do, l.cpu(), m.cpu(), sm_scale=sc, return_dab=True, **okw)[3]
    for dim in (0, 1):
        if ab.shape[dim] == 1:
            ref = ref.sum(dim, keepdim=True)
    assert dab.shape == ab.shape and dab.dtype == ab.dtype
    err = (dab.cpu().double() - ref).abs()
    assert O.rel_l2(dab, ref) <= 1e-2 and bool((err <= 1e-2 * ref.abs().clamp(min=1.0)).all()), float(err.max())


@pytest.mark.parametrize("kind", ["plain", "causal", "alibi"])
def test_bias_gradient_repeats_bit_for_bit(kind):
    """Elements that the last tile of a ragged length shares with the tile before have one writer: the same bits from
    every run, on a grid that fills the chip (4 x 16 heads, 12 kv tiles)."""
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks, scores
    B, H, S, D = 4, 16, 1500, 128
    pair = masks.make_causal_mask_fns(128, 128) if kind == "causal" else None
    sfn = scores.make_alibi_global_score_fn(H) if kind == "alibi" else None
    q, k, v, do = (x.cuda() for x in O.make_inputs(B, H, H, S, S, D, dtype=torch.bfloat16, seed=9))
    ab = torch.randn(B, H, S, S, generator=torch.Generator().manual_seed(1)).cuda()
    for t in (q, k, v, ab):
        t.requires_grad_(True)

    def call():
        o = F.flex_attention(q, k, v, sfn, pair, sm_scale=1.0 if sfn else 1 / math.sqrt(D), ab=ab)
        return torch.autograd.grad(o, (q, k, v, ab), do)
    want = call()
    for _ in range(4):
        for name, a, b in zip(("dq", "dk", "dv", "dab"), call(), want):
            assert torch.equal(a, b), name


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(2, 4, 4, 257, 128), (2, 4, 2, 300, 64)])
@pytest.mark.parametrize("kind", ["alibi", "tile_alibi", "closure", "compiled mask", "documents", "ids per entry"])
def test_bias_gradient_of_every_kernel(kind, B, Hq, Hkv, S, D):
    """The kernels that store the bias gradient are variants of their own per score kind and library: position biases, a
    compiled score function, a compiled mask, documents, segment ids with a row per batch entry."""
    import custom_functors as cf
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks, scores
    sc, pair, sfn, sid, okw = 1 / math.sqrt(D), None, None, None, {}
    if kind == "alibi":
        sfn, okw = scores.make_alibi_global_score_fn(Hq), dict(score_mod=O.score_mod_alibi_global(O.alibi_slopes(Hq)))
    elif kind == "tile_alibi":
        sfn, okw = scores.make_alibi_score_fn(0.02), dict(score_mod=O.score_mod_alibi_tile_local(0.02, 128, 128))
    elif kind == "closure":
        sfn, okw = cf.compiled()["mixed_mod"][0], dict(score_mod=cf.mixed_mod)
    elif kind == "compiled mask":
        i = torch.arange(S)
        pair, okw = cf.compiled()["checker"][1], dict(mask=cf.checker_mask(i, i))
    elif kind == "documents":
        lens = [100, 29, S - 129]
        pair = masks.make_jagged_mask_fns(128, 128, lens)
        okw = dict(causal=True, segment_ids=O.doc_ids_from_lengths(lens))
    else:
        sid = torch.stack([torch.arange(S) * (3 + b) // S for b in range(B)])
        okw = dict(segment_ids=sid)
    ab = torch.randn(1, Hq, S, S, generator=torch.Generator().manual_seed(3))
    okw["ab"] = ab.expand(B, Hq, S, S)
    q, k, v, do = O.make_inputs(B, Hq, Hkv, S, S, D, dtype=torch.bfloat16, seed=S + D)
    qg, kg, vg, abg = [surrounded(x).requires_grad_(True) for x in (q, k, v, ab)]
    o = F.flex_attention(qg, kg, vg, sfn, pair, segment_ids=sid, sm_scale=sc, ab=abg)
    dq, dk, dv, dab = torch.autograd.grad(o, (qg, kg, vg, abg), surrounded(do))
    mf = pair or (None, None)
    with torch.no_grad():
        o2, l, m = F._flex_attention_impl(qg, kg, vg, abg, sid, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], sfn)
    assert torch.equal(o2, o)
    same = same_residual_grads(q, k, v, do, o, l, m, sm_scale=sc, **okw)
    for name, t, r in zip(("dq", "dk", "dv"), (dq, dk, dv), same):
        # (without a causal mask the position bias leaves most of every row's weight on the last keys: their dv sums P dO over
        # all rows, each term with the 2^-9 that P loses in bf16, so the error is of the sum of the terms' sizes, which the
        # tensor's largest entry shows, not of the element that is left after they cancel)
        assert_close(name, t, r, torch.bfloat16, tensor_scale=kind == "alibi")
    ref = O.mha_bwd_reference(q, k, v, o.detach().float().cpu(), do, l.cpu(), m.cpu(), sm_scale=sc, return_dab=True, **okw)[3].sum(0, keepdim=True)
    err = (dab.cpu().double() - ref).abs()
    assert O.rel_l2(dab, ref) <= 1e-2 and bool((err <= 1e-2 * ref.abs().clamp(min=1.0)).all()), float(err.max())
