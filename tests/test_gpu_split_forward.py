"""The plain forward of small grids, whose lists are cut into parts that a second launch puts together (flexattn_fwd_work): one and
several parts, parts that keep nothing of some rows, ragged lengths, grouped heads, both head dimensions, residuals, against the
oracle; and what the call refuses."""
import ctypes as C
import math

import pytest
import torch

from helpers import assert_close
from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,kind", [
    (1, 1, 1, 1024, 1024, "causal"), (1, 2, 1, 1025, 1025, "causal"), (2, 2, 2, 129, 2049, "none"), (1, 4, 2, 300, 1600, "none"),
    (1, 1, 1, 1153, 1153, "window"), (1, 16, 16, 128, 128, "causal"), (1, 1, 1, 128, 8200, "none"), (3, 1, 1, 1100, 1100, "s2")])
def test_split_forward(B, Hq, Hkv, Sq, Sk, kind, D):
    from flex_attention_tpu_amd import _lib, _plans, masks
    from flex_attention_tpu_amd.block_mask import spec_of
    sc = 1 / math.sqrt(D)
    i, j = torch.arange(Sq)[:, None], torch.arange(Sk)[None, :]
    pair, okw = (None, None), {}
    if kind == "causal":
        pair, okw = masks.make_causal_mask_fns(128, 128), dict(causal=True)
    elif kind == "window":   # (a row's keys lie in few of its tile's parts)
        pair, okw = masks.make_causal_sliding_window_mask_fns(128, 128, 40), dict(mask=(j <= i) & (i - j < 40))
    elif kind == "s2":
        pair, okw = masks.make_s2_mask_fns(128, 128, 64, 200), None
        okw = dict(mask=(j <= i) & ((i - j < 64) | (j % 200 == 0)))
    q, k, v, _ = O.make_inputs(B, Hq, Hkv, Sq, Sk, D, dtype=torch.bfloat16, seed=Sq + D)
    qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
    spec = spec_of(*pair)
    assert _plans.takes(qg, kg, spec, sc, _lib.PASS_FWD)
    o, l, m = _plans.forward(qg, kg, vg, spec, sc, True, with_work=True)
    ro, rl, rm = O.mha_reference(q, k, v, sm_scale=sc, save_residuals=True, **okw)
    assert_close("o", o, ro, torch.bfloat16)
    assert_close("lse", m + l.log(), rm + rl.log(), torch.bfloat16)
    for _ in range(3):
        o2, l2, m2 = _plans.forward(qg, kg, vg, spec, sc, True, with_work=True)
        assert torch.equal(o, o2) and torch.equal(l, l2) and torch.equal(m, m2)


def test_bytes_and_refusals():
    from flex_attention_tpu_amd import _lib
    lib = _lib.load()
    q = torch.zeros(1, 1, 2048, 128, dtype=torch.bfloat16, device="cuda")
    p = _lib.FwdParamsC(q=q.data_ptr(), k=q.data_ptr(), v=q.data_ptr(), o=q.data_ptr(), B=1, Hq=1, Hkv=1, Sq=2048, Sk=2048, D=128,
                        dtype=_lib.BF16, sm_scale=1.0)
    assert lib.flexattn_fwd_work_bytes(C.byref(p)) == 0 and lib.flexattn_fwd_work_bytes(None) == 0   # (no block map)
    from flex_attention_tpu_amd.block_mask import build_block_map
    from flex_attention_tpu_amd.masks import MaskSpec
    bm = build_block_map(MaskSpec(), 2048, 2048, *_lib.tile_shape(_lib.PASS_FWD, _lib.BF16, 128), q.device)
    p.map = bm.as_c()
    need = lib.flexattn_fwd_work_bytes(C.byref(p))
    assert need == 4 * 2048 * 130 * 4   # (four parts: eight kv tiles each)
    work = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
    for ptr, n in ((None, need), (work.data_ptr(), need - 1), (work.data_ptr() + 8, need)):
        with pytest.raises(ValueError):
            _lib.check(lib.flexattn_fwd_work(C.byref(p), ptr, n, None), lib)
    p.score.kind = _lib.SCORE_SOFTCAP
    assert lib.flexattn_fwd_work_bytes(C.byref(p)) == 0


@pytest.mark.parametrize("B,Hq,S,D", [(1, 16, 128, 128), (1, 8, 640, 128), (1, 2, 128, 256), (1, 2, 256, 64)])
def test_nothing_to_cut(B, Hq, S, D):
    """Where there is no memory to bring, flexattn_fwd_work is flexattn_fwd: the same bits."""
    from flex_attention_tpu_amd import _lib
    from flex_attention_tpu_amd.block_mask import build_block_map
    from flex_attention_tpu_amd.masks import MaskSpec
    lib = _lib.load()
    q, k, v, _ = (t.cuda() for t in O.make_inputs(B, Hq, Hq, S, S, D, dtype=torch.bfloat16, seed=D))
    bm = build_block_map(MaskSpec(), S, S, *_lib.tile_shape(_lib.PASS_FWD, _lib.BF16, D), q.device)
    got = [[torch.empty_like(q), *torch.empty(2, B, Hq, S, device="cuda")] for _ in range(2)]
    for o, l, m in got:
        p = _lib.FwdParamsC(q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), o=o.data_ptr(), l=l.data_ptr(), m=m.data_ptr(), B=B, Hq=Hq,
                            Hkv=Hq, Sq=S, Sk=S, D=D, dtype=_lib.BF16, sm_scale=D ** -0.5)
        p.map = bm.as_c()
        assert lib.flexattn_fwd_work_bytes(C.byref(p)) == 0
        stream = torch.cuda.current_stream().cuda_stream
        _lib.check(lib.flexattn_fwd_work(C.byref(p), None, 0, stream) if o is got[0][0] else lib.flexattn_fwd(C.byref(p), stream), lib)
    assert all(torch.equal(a, b) for a, b in zip(*got))
