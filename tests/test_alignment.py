"""Operands that are contiguous views at an address that is no multiple of 16 bytes (a slice of a flat buffer): the entry
points take them and return what they return for aligned copies, bit for bit; the C calls whose kernels read the caller's
tensors in 16-byte pieces at every length refuse them."""
import ctypes as C
import math

import pytest
import torch

from flex_attention_tpu_amd import _lib
from oracle import mha_oracle as O


def shifted(t, by):
    """A contiguous copy of the GPU tensor `t`, `by` elements behind an aligned address."""
    big = torch.full((t.numel() + 64,), float("nan"), dtype=t.dtype, device=t.device)
    out = big[by:by + t.numel()].view(t.shape)
    out.copy_(t)
    return out


def test_aligned():
    from flex_attention_tpu_amd._common import aligned
    big = torch.arange(64, dtype=torch.bfloat16)
    at = next(i for i in range(8) if big[i:].data_ptr() % 16 == 0)
    view = big[at:at + 16]
    assert aligned(view) is view
    for by in range(1, 8):
        view = big[at + by:at + by + 16]
        out = aligned(view)
        assert out.data_ptr() % 16 == 0 and torch.equal(out, view)


def test_c_calls_refuse_unaligned_operands(lib):
    ptr = (C.c_uint8 * 64)()
    base = (C.addressof(ptr) + 15) // 16 * 16
    for D, pad, fn in ((64, 0, lib.flexattn_fwd), (128, 5, lib.flexattn_fwd)):
        p = _lib.FwdParamsC(q=base, k=base + 2, v=base, o=base, B=1, Hq=1, Hkv=1, Sq=128, Sk=128, D=D, dtype=_lib.BF16, sm_scale=1.0, pad=pad)
        assert fn(C.byref(p), None) == _lib.EINVAL and b"16 bytes" in lib.flexattn_last_error_string()
    p = _lib.FwdParamsC(q=base, k=base, v=base + 8, o=base, B=1, Hq=1, Hkv=1, Sq=1, Sk=256, D=128, dtype=_lib.BF16, sm_scale=1.0)
    assert lib.flexattn_fwd_decode(C.byref(p), None, 0, None) == _lib.EINVAL and b"16 bytes" in lib.flexattn_last_error_string()
    p = _lib.BwdParamsC(q=base, k=base, v=base, dout=base + 4, l=base, m=base, delta=base, dq=base, B=1, Hq=1, Hkv=1, Sq=128, Sk=128, D=128,
                        dtype=_lib.BF16, sm_scale=1.0, pad=5)
    assert lib.flexattn_bwd_dq(C.byref(p), None) == _lib.EINVAL and b"16 bytes" in lib.flexattn_last_error_string()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,dtype,D,Sq,Sk", [
    ("plain", torch.bfloat16, 128, 256, 256), ("plain", torch.bfloat16, 128, 321, 257), ("plain", torch.bfloat16, 64, 256, 384),
    ("plain", torch.bfloat16, 64, 3, 515), ("plain", torch.bfloat16, 128, 3, 515), ("plain", torch.bfloat16, 256, 321, 321), ("softcap", torch.bfloat16, 128, 321, 321),
    ("bias", torch.bfloat16, 128, 257, 257), ("plain", torch.float32, 64, 321, 257), ("plain", torch.float32, 128, 256, 256)])
def test_unaligned_views(kind, dtype, D, Sq, Sk):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import scores
    B, H, sc = 2, 2, 1 / math.sqrt(D)
    sfn = scores.make_softcap_score_fn(5.0) if kind == "softcap" else None
    q, k, v, do = (x.cuda() for x in O.make_inputs(B, H, H, Sq, Sk, D, dtype=dtype, seed=Sq))
    ab = torch.randn(1, H, Sq, Sk, generator=torch.Generator().manual_seed(1)).cuda() if kind == "bias" else None

    def call(*ts):
        *ts, do_, ab_ = ts
        leaves = [t.requires_grad_(True) for t in ts] + ([ab_.requires_grad_(True)] if ab_ is not None else [])
        o = F.flex_attention(*ts, sfn, None, sm_scale=sc, ab=ab_)
        return (o.detach(), *torch.autograd.grad(o, leaves, do_))

    def passes(q, k, v, do, ab):
        with torch.no_grad():
            o, l, m = F._flex_attention_impl(q, k, v, ab, None, True, False, sc, 1, 128, 128, 128, False, None, None, sfn)
            o = shifted(o, 1) if q.data_ptr() % 16 else o
            kw = dict(block_b=1, block_q=128, block_k_major=128, block_k=128, sm_scale=sc, debug=False, score_fn=sfn)
            dq, d = F.flex_attention_bwd_dq(q, k, v, ab, None, l, m, o, do, None, return_delta=True, **kw)
            d2 = F.compute_delta(o, do)
            return (o, l, m, dq, d, d2, *F.flash_attention_bwd_dkv(k, v, q, ab, None, l, m, d, do, block_q_major=128, causal=False, **kw))
    for fn in (call, passes):
        want = fn(q, k, v, do, ab)
        for by in (1, 3):
            got = fn(*(shifted(t.detach(), by) for t in (q, k, v, do)), shifted(ab.detach(), by) if ab is not None else None)
            for i, (a, b) in enumerate(zip(got, want)):
                assert torch.equal(a, b), (fn.__name__, by, i)
