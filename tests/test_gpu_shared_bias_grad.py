"""The gradient of a bias that several (batch, head) pairs share, from the pass that sums over them: edges of tiles, every way a
bias broadcasts, masks whose tiles are partial or empty, documents per batch entry, grouped heads, bf16 biases, against the oracle
on the kernels' own forward.  Tolerances as in test_gpu_bias_grad: values are P (dP - delta) summed over the pairs, 1e-2 of a value
where that exceeds 1."""
import math
import types

import pytest
import torch

from helpers import assert_close, same_residual_grads
from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["plain", "causal", "window", "ids per entry", "bf16 bias"])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,ab_shape", [
    (2, 34, 34, 129, 257, 128, "1h"), (3, 34, 17, 255, 383, 64, "1h"), (2, 50, 50, 256, 256, 128, "1h"),
    (34, 3, 1, 321, 130, 128, "b1"), (2, 2, 2, 1800, 1700, 96, "11"), (1, 2, 1, 1792, 1920, 128, "11")])
def test_shared_bias_gradient(B, Hq, Hkv, Sq, Sk, D, ab_shape, kind, monkeypatch):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _lib, masks
    sc, pair, sid, okw = 1 / math.sqrt(D), None, None, {}
    i, j = torch.arange(Sq)[:, None], torch.arange(Sk)[None, :]
    if kind == "causal":
        pair, okw = masks.make_causal_mask_fns(128, 128), dict(causal=True)
    elif kind == "window":   # (tiles that no pair keeps: their gradient is zero)
        window = 100 + max(0, Sq - Sk)   # (every query keeps a key)
        pair, okw = masks.make_causal_sliding_window_mask_fns(128, 128, window), dict(mask=(j <= i) & (i - j < window))
    elif kind == "ids per entry":
        ids = [torch.stack([torch.arange(S) * (2 + b) // S for b in range(B)]) for S in (Sq, Sk)]
        sid = types.SimpleNamespace(q=ids[0], kv=ids[1])
        okw = dict(mask=ids[0][:, :, None] == ids[1][:, None, :])
    ab = torch.randn(B if ab_shape[0] == "b" else 1, Hq if ab_shape[1] == "h" else 1, Sq, Sk, generator=torch.Generator().manual_seed(3))
    if kind == "bf16 bias":
        ab = ab.bfloat16()
    okw["ab"] = ab.float().expand(B, Hq, Sq, Sk)
    q, k, v, do = O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=torch.bfloat16, seed=Sq + D)
    qg, kg, vg, abg = [x.cuda().requires_grad_(True) for x in (q, k, v, ab)]
    lib, launched = _lib.load(), []
    real = lib.flexattn_bwd_dab
    monkeypatch.setattr(lib, "flexattn_bwd_dab", lambda *a: launched.append(1) or real(*a))
    o = F.flex_attention(qg, kg, vg, None, pair, segment_ids=sid, sm_scale=sc, ab=abg)
    dq, dk, dv, dab = torch.autograd.grad(o, (qg, kg, vg, abg), do.cuda())
    assert launched
    mf = pair or (None, None)
    with torch.no_grad():
        _, l, m = F._flex_attention_impl(qg, kg, vg, abg, sid, True, False, sc, 1, 128, 128, 128, False, mf[1], mf[0], None)
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
    for _ in range(3):   # (one writer per element, pairs in order: the same bits from every run)
        o = F.flex_attention(qg, kg, vg, None, pair, segment_ids=sid, sm_scale=sc, ab=abg)
        assert torch.equal(torch.autograd.grad(o, (qg, kg, vg, abg), do.cuda())[3], dab)
