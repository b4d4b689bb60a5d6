"""Sequence lengths around the edges of the kernels' tiles: the last tile of a length that is no multiple of the tile
starts early, so that nothing outside a head's rows is read.  The inputs lie inside larger arrays of NaN: a row from
beyond a tensor would show in every result it touches.  Tolerances: helpers.assert_close."""
import math

import pytest
import torch

from helpers import assert_close, same_residual_grads
from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def surrounded(t, pad=512):
    """A contiguous copy of `t` on the GPU with `pad` elements of NaN in front of and behind it."""
    big = torch.full((t.numel() + 2 * pad,), float("nan"), dtype=t.dtype, device=DEV)
    out = big[pad:pad + t.numel()].view(t.shape)
    out.copy_(t)
    return out


KINDS = {
    # name: (Hq, Hkv, D, dtype, compiled_loop)
    "stream": (2, 2, 128, torch.bfloat16, False),
    "stream_causal_gqa": (4, 2, 128, torch.bfloat16, False),
    "stream_alibi_window": (2, 2, 128, torch.bfloat16, False),
    "stream_softcap_documents": (2, 1, 128, torch.bfloat16, False),
    "stream_unsorted_ids": (2, 2, 128, torch.bfloat16, False),
    "compiled_causal": (2, 1, 128, torch.bfloat16, True),
    "compiled_documents": (2, 2, 128, torch.bfloat16, True),
    "bias": (2, 2, 128, torch.bfloat16, False),
    "d256_causal": (2, 1, 256, torch.bfloat16, False),
    "d256": (1, 1, 256, torch.bfloat16, False),
    "d64": (2, 1, 64, torch.bfloat16, False),
    "d64_causal": (2, 2, 64, torch.bfloat16, False),
    "d64_bias": (2, 2, 64, torch.bfloat16, False),
    "fp32_causal": (2, 1, 64, torch.float32, False),
    "fp32_d128": (2, 2, 128, torch.float32, False),
    "fp32_bias": (2, 2, 64, torch.float32, False),
    "fp32_scalar": (2, 1, 64, torch.float32, True),
}
LENGTHS = [(128, 129), (129, 191), (193, 128), (255, 257), (385, 321), (300, 640)]


@pytest.mark.parametrize("Sq,Sk", LENGTHS)
@pytest.mark.parametrize("kind", KINDS)
def test_lengths_around_the_tiles(kind, Sq, Sk):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import masks, scores
    Hq, Hkv, D, dtype, loop = KINDS[kind]
    B, sc = 2, 1 / math.sqrt(D)
    mf, sfn, okw, sid, ab = (None, None), None, {}, None, None
    if "causal" in kind:
        mf, okw = masks.make_causal_mask_fns(128, 128), dict(causal=True)
    if "alibi" in kind:
        W = 150 + max(0, Sq - Sk)      # (every query keeps a key)
        mf = masks.make_sliding_window_mask_fns(128, 128, W)
        sfn = scores.make_alibi_global_score_fn(Hq)
        okw = dict(window_size=W, score_mod=O.score_mod_alibi_global(O.alibi_slopes(Hq)))
    if "documents" in kind or "unsorted" in kind:
        n = 3
        ids_q, ids_k = (torch.arange(S) * n // S for S in (Sq, Sk))
        if "unsorted" in kind:
            ids_k = ids_k.flip(0)
        import types
        sid = types.SimpleNamespace(q=ids_q, kv=ids_k)
        okw = dict(mask=ids_q[:, None] == ids_k[None, :])
    if "softcap" in kind:
        sfn = scores.make_softcap_score_fn(5.0)
        okw["score_mod"] = O.score_mod_softcap(5.0)
    if "bias" in kind:
        ab = torch.randn(1, Hq, Sq, Sk, generator=torch.Generator().manual_seed(3))
        okw["ab"] = ab.expand(B, Hq, Sq, Sk)
    q, k, v, do = O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=dtype, seed=11)
    ro, rl, rm = O.mha_reference(q, k, v, sm_scale=sc, save_residuals=True, **okw)
    qg, kg, vg, dog = [surrounded(x) for x in (q, k, v, do)]
    abg = surrounded(ab) if ab is not None else None
    o, l, m = F._flex_attention_impl(qg, kg, vg, abg, sid, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], sfn,
                                     compiled_loop=loop)
    assert_close("o", o, ro, dtype)
    assert_close("lse", m + l.log(), rm + rl.log(), dtype)
    l, m, os_ = surrounded(l), surrounded(m), surrounded(o)
    d = surrounded(F.compute_delta(os_, dog))
    kw = dict(block_q=128, block_k_major=128, block_k=128, sm_scale=sc, debug=False, score_fn=sfn, mask_fn=mf[0],
              block_mask_fn=mf[1], compiled_loop=loop)
    dq = F.flex_attention_bwd_dq(qg, kg, vg, abg, sid, l, m, os_, dog, d, block_b=1, return_dab=ab is not None, **kw)
    if ab is not None:
        dq, dab = dq
        rdab = O.mha_bwd_reference(q, k, v, o.float().cpu(), do, l.cpu(), m.cpu(), sm_scale=sc, return_dab=True, **okw)[3]
        rdab = rdab.sum(0, keepdim=True)
        assert dab.shape == ab.shape
        # (dab is P (dP - delta): the bound of its values, relative where they exceed 1)
        rel = 1e-5 if dtype == torch.float32 else 1e-2
        err = (dab.cpu().double() - rdab).abs()
        assert O.rel_l2(dab, rdab) <= rel and bool((err <= rel * rdab.abs().clamp(min=1.0)).all()), float(err.max())
    dk, dv, ds = F.flash_attention_bwd_dkv(kg, vg, qg, abg, sid, l, m, d, dog, block_b=1, block_q_major=128, causal=False,
                                           return_ds=True, **kw)
    same = same_residual_grads(q, k, v, do, o, l, m, sm_scale=sc, **okw)
    got = [("dq", dq, same[0]), ("dk", dk, same[1]), ("dv", dv, same[2])]
    if ds is not None:   # (the dk/dv pass hands dS over: the dq pass from it, and dk, dv without the export)
        dk2, dv2 = F.flash_attention_bwd_dkv(kg, vg, qg, abg, sid, l, m, d, dog, block_b=1, block_q_major=128, causal=False, **kw)
        assert torch.equal(dk2, dk) and torch.equal(dv2, dv)
        got.append(("dq from dS", F.flex_attention_bwd_dq(qg, kg, vg, abg, sid, l, m, os_, dog, d, block_b=1, ds=ds, **kw), same[0]))
    for name, t, r in got:
        assert_close(name, t, r, dtype)
