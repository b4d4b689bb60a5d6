"""The forward of a few query rows against long keys (fwd_decode.hip) at the edges of its tiles, row blocks and splits:
against the dense oracle, with NaN around every operand.  Tolerances: helpers.assert_close."""
import math

import pytest
import torch

from helpers import assert_close
from oracle import mha_oracle as O
from test_gpu_ragged import surrounded

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows per kv head 1, 31 .. 33, 64, 65, 128; keys around the tiles (32 and 64), fewer tiles than waves, many splits
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk", [
    (1, 1, 1, 1, 128), (2, 4, 1, 1, 129), (1, 8, 2, 2, 191), (3, 2, 2, 31, 160), (1, 4, 4, 32, 1000), (2, 3, 1, 11, 257),
    (1, 32, 1, 2, 4001), (1, 5, 1, 13, 640), (1, 8, 1, 16, 2048), (40, 8, 8, 1, 515), (1, 2, 1, 1, 32768)])
@pytest.mark.parametrize("D", [64, 128, 40])
def test_decode(B, Hq, Hkv, Sq, Sk, D):
    import flex_attention_tpu_amd as F
    from flex_attention_tpu_amd import _lib
    g = torch.Generator().manual_seed(Sk * 131 + Sq + D)
    q, k, v = (torch.randn(B, h, s, D, generator=g).bfloat16() for h, s in ((Hq, Sq), (Hkv, Sk), (Hkv, Sk)))
    k[0, 0, -1] *= 3.0     # (the last key weighs in: a lost or doubled last tile shows)
    sc = 1 / math.sqrt(D)
    p = _lib.FwdParamsC(B=B, Hq=Hq, Hkv=Hkv, Sq=Sq, Sk=Sk, D=64 if D <= 64 else 128, dtype=_lib.BF16)
    assert _lib.load().flexattn_fwd_decode_bytes(p) >= 0
    qg, kg, vg = (surrounded(x) for x in (q, k, v))
    o, l, m = F._flex_attention_impl(qg, kg, vg, None, None, True, False, sc, 1, 128, 128, 128, False, None, None, None)
    ro, rl, rm = O.mha_reference(q, k, v, sm_scale=sc, save_residuals=True)
    assert_close("o", o, ro, torch.bfloat16)
    assert_close("lse", m + l.log(), rm + rl.log(), torch.float32, tensor_scale=True)
    assert torch.equal(F.flex_attention(qg, kg, vg, sm_scale=sc), o)
