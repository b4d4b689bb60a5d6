"""End-to-end differentiable flex attention: forward + delta + dq + dk/dv behind one
``torch.autograd.Function``.

The reference wires its three kernels together with ``jax.custom_vjp`` (upstream copy in
jax_exp.py:207-321: ``_flash_attention`` / ``_flash_attention_fwd`` saves ``(q, k, v, ab,
segment_ids, o, l, m)``; ``_flash_attention_bwd`` computes ``di = sum(o * do, -1)`` in float32 and
calls the dk/dv and the dq kernels).  This is the same wiring on the HIP entry points of this
package, with the flex arguments (``score_fn``, ``mask_fn`` / ``block_mask_fn``) of
flex_attention_kernel.py:66-83 carried through.
"""
from __future__ import annotations

import ctypes as C
import math
from typing import Callable, Optional, Tuple

import torch

from . import _lib, _plans
from ._common import aligned, call_head_dim, check_blocks, check_qkv, check_rows, on_device, stream_of, tagged_closures
from .block_mask import spec_of
from .flex_attention_dkv_kernel import flash_attention_bwd_dkv
from .flex_attention_dq_bwd import compute_delta, ds_exchange_pays, flex_attention_bwd_dq
from .flex_attention_kernel import _CAUSAL, _flex_attention_impl


def _hands_ds_over(q, k, ab, segment_ids, sm_scale, score_fn, mask_fn, block_mask_fn, want_dab) -> bool:
    """Whether a bf16 backward that wants every gradient hands dS from the dk/dv pass to the dq pass (DsBlocks in
    flex_attention_dq_bwd.py).  The buffer holds one 32 KB block per query head and kept pair of 128 x 128 tiles (what the
    mask skips takes no room)."""
    D = q.shape[-1]
    if want_dab:   # (the bias gradient is the fp32 dS that the dk/dv pass rounds for the hand-over: one pass makes both, and the dq
        return D <= 128   # pass is one product instead of three; B=4, H=16, S=1500, forward and backward: 1.19 -> 1.03 ms)
    if ab is not None:
        return False
    # (at head dimension 256 always: the recomputing dq pass costs three products of twice the depth.  On B=4, H=16,
    # S=4096, causal, forward and backward: 3.61 -> 3.08 ms.  Not at the head dimension 64 kernels, which hand nothing over:
    # recomputing there beats the hand-over on 128 padded columns also where that pays at 128 columns; documents, B=4, H=16,
    # S=4096: 1.40 -> 0.71 ms, GQA 4:1, S=16384: 1.81 -> 1.16 ms; causal window 1025, B=2, H=16, S=8192: 0.97 -> 0.46 ms.)
    return ((D > 128 or ds_exchange_pays(score_fn, mask_fn, segment_ids)) and
            call_head_dim(_lib.PASS_DKV, D, q.dtype, sm_scale, score_fn, ab, spec_of(mask_fn, block_mask_fn), q.shape[2], k.shape[2]) != 64)


def _bwd_with_ds(q, k, v, ab, segment_ids, l, m, o, do, want_dab, block_q, block_k, sm_scale, causal, score_fn, mask_fn, block_mask_fn):
    """The gradients of q, k, v and the bias (or None) as the autograd function returns them, with dS handed from the dk/dv
    pass to the dq pass; where the dk/dv entry point declines to (no room for the buffer, kernels that exchange nothing),
    the dq pass recomputes."""
    kw = dict(block_b=1, block_q=block_q, block_k_major=block_k, block_k=block_k, sm_scale=sm_scale, causal=causal, debug=False,
              score_fn=score_fn, mask_fn=mask_fn, block_mask_fn=block_mask_fn)
    di = compute_delta(o, do)
    dk, dv, ds, *dab = flash_attention_bwd_dkv(k, v, q, ab, segment_ids, l, m, di, do, block_q_major=block_q, return_ds=True,
                                               _wide_ds=not want_dab, _dab=want_dab, **kw)
    if ds is None and want_dab:
        dq, dab = flex_attention_bwd_dq(q, k, v, ab, segment_ids, l, m, o, do, di, return_dab=True, **kw)
        return dq, dk, dv, dab, None
    dq = flex_attention_bwd_dq(q, k, v, ab, segment_ids, l, m, o, do, di, ds=ds, **kw)
    return dq, dk, dv, (dab[0] if want_dab else None), None


def flex_attention_bwd(q, k, v, ab, segment_ids, l, m, o, do, *, block_q, block_k, sm_scale, causal=False, score_fn=None,
                       mask_fn=None, block_mask_fn=None, compiled_loop=False):
    """(dq, dk, dv) of one backward: delta = sum(o * do), the dq pass and the dk/dv pass (the sequence of the
    reference's custom_vjp wiring, jax_exp.py:276-321) from one call through the C ABI (flexattn_bwd): small
    problems are bound by the host's path to a launch.  No dS hand-over (see flash_attention_bwd_dkv(return_ds=True) for that) and no bias
    gradient (flex_attention_bwd_dq(return_dab=True))."""
    if score_fn is None and ab is None and segment_ids is None and not compiled_loop:
        B, Hq, _, Sq, Sk, _ = check_qkv(q, k, v, do, o)
        check_blocks(Sq, Sk, block_q=block_q, block_k_major=block_k, block_k=block_k)
        check_rows("l", l, B, Hq, Sq, q.device)
        check_rows("m", m, B, Hq, Sq, q.device)
        _, mask_fn, block_mask_fn = tagged_closures(None, mask_fn, block_mask_fn, block_q, block_k)
        spec = spec_of(mask_fn, block_mask_fn)
        if causal:
            spec = spec.combine(_CAUSAL)
        if _plans.takes(q, k, spec, sm_scale, _lib.PASS_DQ, _lib.PASS_DKV):
            return _plans.backward(q, k, v, l, m, o, do, spec, float(sm_scale))
    if (q.data_ptr() | k.data_ptr() | v.data_ptr() | do.data_ptr()) % 16:   # (the two passes share them)
        q, k, v, do = aligned(q), aligned(k), aligned(v), aligned(do)
    kw = dict(sm_scale=sm_scale, debug=False, score_fn=score_fn, mask_fn=mask_fn, block_mask_fn=block_mask_fn,
              compiled_loop=compiled_loop)
    dq_call = flex_attention_bwd_dq(q, k, v, ab, segment_ids, l, m, o, do, None, block_b=1, block_q=block_q,
                                    block_k_major=block_k, block_k=block_k, causal=causal, return_delta=True, _defer=True, **kw)
    dkv_call = None
    if dq_call is not None and dq_call["delta"] is not None:
        dkv_call = flash_attention_bwd_dkv(k, v, q, ab, segment_ids, l, m, dq_call["delta"], do, block_b=1, block_q=block_q,
                                           block_q_major=block_q, block_k_major=block_k, block_k=block_k, causal=causal,
                                           _defer=True, **kw)
    if dkv_call is None:   # (padded shapes, ids per batch entry: the passes one after the other)
        dq, di = flex_attention_bwd_dq(q, k, v, ab, segment_ids, l, m, o, do, None, block_b=1, block_q=block_q,
                                       block_k_major=block_k, block_k=block_k, causal=causal, return_delta=True, **kw)
        dk, dv = flash_attention_bwd_dkv(k, v, q, ab, segment_ids, l, m, di, do, block_b=1, block_q=block_q,
                                         block_q_major=block_q, block_k_major=block_k, block_k=block_k, causal=causal, **kw)
        return dq, dk, dv
    lib = dq_call["lib"]
    with on_device(q.device):
        _lib.check(lib.flexattn_bwd(C.byref(dq_call["params"]), C.byref(dkv_call["params"]), stream_of(q)), lib)
    dq, _ = dq_call["finish"]()
    dk, dv = dkv_call["finish"]()
    return dq, dk, dv


class _FlexAttention(torch.autograd.Function):
    """o = softmax(mask(score_mod(sm_scale q k^T))) v with the saved statistics (l, m) for the backward."""

    @staticmethod
    def forward(ctx, q, k, v, ab, opts):
        score_fn, mask_fn, block_mask_fn, segment_ids, causal, sm_scale, block_q, block_k = opts
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
        o, l, m = _flex_attention_impl(q, k, v, ab, segment_ids, True, causal, sm_scale, 1, block_q, block_k, block_k,
                                       False, block_mask_fn, mask_fn, score_fn, _with_work=True)
        ctx.save_for_backward(q, k, v, o, l, m, *([ab] if ab is not None else []))
        ctx.opts = opts
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, l, m, *rest = ctx.saved_tensors
        ab = rest[0] if rest else None
        score_fn, mask_fn, block_mask_fn, segment_ids, causal, sm_scale, block_q, block_k = ctx.opts
        want_dab = ab is not None and ctx.needs_input_grad[3]
        do = do.contiguous()
        dq = dk = dv = dab = None
        want_dkv = ctx.needs_input_grad[1] or ctx.needs_input_grad[2]
        want_dq = ctx.needs_input_grad[0] or want_dab
        if want_dkv and ctx.needs_input_grad[0]:
            if q.dtype is torch.bfloat16 and _hands_ds_over(q, k, ab, segment_ids, sm_scale, score_fn, mask_fn, block_mask_fn, want_dab):
                try:
                    return _bwd_with_ds(q, k, v, ab, segment_ids, l, m, o, do, want_dab, block_q, block_k, sm_scale, causal, score_fn,
                                        mask_fn, block_mask_fn)
                except torch.cuda.OutOfMemoryError:
                    pass   # (beside the dS buffer there was no room for the rest: below nothing needs one)
            if not want_dab:
                dq, dk, dv = flex_attention_bwd(q, k, v, ab, segment_ids, l, m, o, do, block_q=block_q, block_k=block_k,
                                                sm_scale=sm_scale, causal=causal, score_fn=score_fn, mask_fn=mask_fn,
                                                block_mask_fn=block_mask_fn)
                return dq, dk, dv, None, None
        kw = dict(block_b=1, block_q=block_q, block_k=block_k, block_k_major=block_k, sm_scale=sm_scale, causal=causal, debug=False,
                  score_fn=score_fn, mask_fn=mask_fn, block_mask_fn=block_mask_fn)
        # di = sum(o * do), float32 [B, H, Sq] (jax_exp.py:276-278): taken by the dq pass itself where that pass runs
        # first, else by its own launch
        di = None
        if want_dq:
            dq = flex_attention_bwd_dq(q, k, v, ab, segment_ids, l, m, o, do, None, return_dab=want_dab, return_delta=not want_dab, **kw)
            if want_dab:
                dq, dab = dq
            else:
                dq, di = dq
        if want_dkv:
            if di is None:
                di = compute_delta(o, do)
            dk, dv = flash_attention_bwd_dkv(k, v, q, ab, segment_ids, l, m, di, do, block_q_major=block_q, **kw)
        return dq if ctx.needs_input_grad[0] else None, dk, dv, dab, None


def flex_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, score_fn: Optional[Callable] = None,
                   mask_fns: Optional[Tuple[Callable, Callable]] = None, *, segment_ids=None, causal: bool = False,
                   sm_scale: Optional[float] = None, block_q: int = 128, block_k: int = 128,
                   ab: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Differentiable flex attention on ``[B, H, S, D]`` GPU tensors (k, v may have fewer heads: GQA).

    ``score_fn``   closure from ``scores`` (or ``util.make_jax_score_fn`` / ``compiler.compile_score_mod``), a plain
                   Python function ``f(q_tile, k_tile)`` or ``f(s, b, h, q_idx, kv_idx)`` (compiled at first use), or None
    ``mask_fns``   ``(mask_fn, block_mask_fn)`` pair from ``masks`` (or ``compiler.compile_mask_fn``), a pair whose
                   ``mask_fn(q_idx, k_idx)`` is a plain Python function (compiled at first use, the block closure
                   derived from it), such a function alone, or None
    ``segment_ids`` / ``causal``   as in the three entry points (ANDed with ``mask_fns``)
    ``sm_scale``   default 1 / sqrt(D)
    ``ab``         additive bias on the logits, [B or 1, H or 1, Sq, Sk]; a bias that requires grad receives
                   dab = P (dP - delta), summed over the dimensions it broadcasts (the output the reference declares
                   next to dk, dv, flash_attention_dkv_bwd.py:103-107,130-138)
    Gradients flow to q, k, v and ab (``torch.autograd.grad`` / ``.backward()``); higher-order
    differentiation is not supported, as in the reference (jax_exp.py:243-244).
    """
    if torch.compiler.is_dynamo_compiling():   # (torch.compile makes the call between its graphs: block maps, plans and launches are no part of one)
        return torch.compiler.disable(_uncompiled)(q, k, v, score_fn, mask_fns, segment_ids=segment_ids, causal=causal, sm_scale=sm_scale,
                                                   block_q=block_q, block_k=block_k, ab=ab)
    if sm_scale is None:
        sm_scale = 1.0 / math.sqrt(q.shape[-1])
    if callable(mask_fns):   # (a bare mask function instead of a pair)
        mask_fn, block_mask_fn = mask_fns, None
    else:
        mask_fn, block_mask_fn = mask_fns if mask_fns is not None else (None, None)
    score_fn, mask_fn, block_mask_fn = tagged_closures(score_fn, mask_fn, block_mask_fn, block_q, block_k)
    if score_fn is None and ab is None and segment_ids is None and _plans.long_and_narrow(q):
        known = getattr(mask_fn if mask_fn is not None else block_mask_fn, "spec", None)
        # (in the order of their cost: documents, compiled masks and windows pay for no further look)
        if (known is None or (known.doc_ids is None and known.custom is None and
                              not (q.dtype is torch.bfloat16 and q.size(3) > 64 and ds_exchange_pays(None, mask_fn)))) and _plans.ordinary(q, k, v):
            spec = spec_of(mask_fn, block_mask_fn)
            if causal:
                spec = spec.combine(_CAUSAL)

            def prepared(q, k, v, spec):
                B, Hq, Hkv, Sq, Sk, D = check_qkv(q, k, v)
                check_blocks(Sq, Sk, block_q=block_q, block_k_major=block_k, block_k=block_k)
                return (_plans.takes(q, k, spec, sm_scale, _lib.PASS_FWD, _lib.PASS_DQ, _lib.PASS_DKV) and
                        not (q.dtype is torch.bfloat16 and _hands_ds_over(q, k, None, None, sm_scale, None, mask_fn, block_mask_fn, False)))
            o = _plans.attend(q, k, v, spec, float(sm_scale), block_q, block_k, prepared)
            if o is not None:
                return o
    opts = (score_fn, mask_fn, block_mask_fn, segment_ids, bool(causal), float(sm_scale), int(block_q), int(block_k))
    return _FlexAttention.apply(q, k, v, ab, opts)


def _uncompiled(*args, **kwargs):
    return flex_attention(*args, **kwargs)
