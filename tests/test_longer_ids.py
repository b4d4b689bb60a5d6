"""Document ids that cover more positions than a call of ragged lengths has: the call takes the first ones, also where every
batch entry has ids of its own."""
import numpy as np
import pytest
import torch

from flex_attention_tpu_amd import _lib
from flex_attention_tpu_amd._common import resolve_mask
from flex_attention_tpu_amd.masks import DocIds, MaskSpec
from oracle import mha_oracle as O


def tagged(ids):
    def mask_fn(q_idx, k_idx):
        raise AssertionError("never called")
    mask_fn.spec = MaskSpec(flags=_lib.MASK_DOC, doc_ids=DocIds(ids))
    return mask_fn


@pytest.mark.parametrize("rows", [None, 2])
@pytest.mark.parametrize("Sq,Sk", [(321, 321), (129, 321), (256, 257)])
def test_ids_are_cut_to_a_ragged_call(rows, Sq, Sk):
    ids = np.arange(400) // 50
    if rows:
        ids = np.stack([ids, np.arange(400) // 70])
    spec = resolve_mask(tagged(ids), None, False, None, Sq, Sk, Sq, Sk)
    ids_k = spec.doc_ids_k if spec.doc_ids_k is not None else spec.doc_ids
    assert np.array_equal(spec.doc_ids.array, ids[..., :Sq]) and np.array_equal(ids_k.array, ids[..., :Sk])
    assert resolve_mask(tagged(ids[..., :Sq]), None, False, None, Sq, Sq, Sq, Sq) == MaskSpec(flags=_lib.MASK_DOC, doc_ids=DocIds(ids[..., :Sq]))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [None, 2])
def test_ids_longer_than_a_ragged_call(rows):
    import flex_attention_tpu_amd as F
    B, H, S, D = 2, 2, 321, 128
    ids = np.arange(400) // 50
    if rows:
        ids = np.stack([ids, np.arange(400) // 70])
    q, k, v, do = (x.cuda().requires_grad_(True) for x in O.make_inputs(B, H, H, S, S, D, dtype=torch.bfloat16, seed=1))

    def call(ids):
        o = F.flex_attention(q, k, v, None, (tagged(ids), None))
        return (o, *torch.autograd.grad(o, (q, k, v), do))
    assert all(torch.equal(a, b) for a, b in zip(call(ids), call(ids[..., :S])))
