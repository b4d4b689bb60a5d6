"""Prepared launches of the plain calls (no score function, bias or document ids, lengths of at least a tile, a head
dimension that needs no padding): what their parameter blocks hold besides pointers depends on shapes, mask and scale
alone and is assembled once per combination.

Small problems are bound by the host's path to a launch: forward and backward of B=1, H=4, S=512, D=64 in float32 keep
the GPU busy for 83 us and took the host 221 us, 154 us this way.  A prepared call checks its tensors as every other call does, takes the
template, writes its pointers into a copy of its own and launches: nothing of a call's tensors is kept.  `attend` is the same
with the autograd function, the allocations and the launches in C++ (csrc/host_path.cpp): 81 us, the kernels' own time.
"""
from __future__ import annotations

import ctypes as C
import struct
import weakref
from typing import Optional

import torch

from . import _lib
from ._common import aligned, call_head_dim, dtype_code, on_device, stream_of, tile_lengths
from .block_mask import LRU, build_block_map, mask_spec_c
from .masks import MaskSpec

_plans = LRU(64)   # (pass, q shape, k shape, dtype, device, mask, scale) -> _Plan; bounded, holds no device memory
_FWD_POINTERS = struct.Struct("6P")     # q, k, v, o, l, m
_BWD_POINTERS = struct.Struct("10P")    # q, k, v, dout, l, m, delta, dq, dk, dv


class _Plan:
    """Parameter templates (bytes) of one combination and weak references to the block maps they point at: the maps
    belong to their own bounded cache, and a plan whose map has been dropped there is made again."""
    __slots__ = ("templates", "maps", "work_bytes")

    def __init__(self, templates, maps):
        self.templates, self.maps = templates, tuple(weakref.ref(bm) for bm in maps)
        self.work_bytes = None   # (of the forward, asked at first use)


def _template(cls, pass_id, q, k, spec, sm_scale):
    B, Hq, Sq, D = q.shape
    _, Hkv, Sk, _ = k.shape
    code = dtype_code(q)
    bq, bk = _lib.tile_shape(pass_id, code, D)
    bm = build_block_map(spec, Sq, Sk, bq, bk, q.device, ragged=True)
    Sq_c, Sk_c, pad = tile_lengths(bm)
    p = cls(B=B, Hq=Hq, Hkv=Hkv, Sq=Sq_c, Sk=Sk_c, D=D, dtype=code, sm_scale=float(sm_scale), pad=pad,
            score=_lib.ScoreSpecC(_lib.SCORE_NONE, 0.0, 0.0, 1, 1, 0, None), mask=mask_spec_c(spec, Sq, Sk, q.device), map=bm.as_c())
    return bytes(p), bm


def _keep(plans, key, plan, maps):
    """Adds a plan to its cache, unless it refers to a map that a captured call has built: only that call's graph fills it."""
    if not any(bm.captured for bm in maps):
        plans.put(key, plan)


def _plan(key, q, k, spec, sm_scale, cls, passes):
    """(plan, block maps) of a combination; the caller holds the maps until its launch is out."""
    plan = _plans.get(key)
    maps = [ref() for ref in plan.maps] if plan is not None else (None,)
    if None in maps:
        templates, maps = zip(*(_template(cls, pass_id, q, k, spec, sm_scale) for pass_id in passes))
        plan = _Plan(templates, maps)
        _keep(_plans, key, plan, maps)
    for bm in maps:   # (a map built on another stream: this one waits for it)
        bm.wait_ready(q.device)
    return plan, maps


_attend_plans = LRU(64)   # (shapes, dtype, device, mask, scale, blocks) -> (C++ plan, weak references to its block maps), or False
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def long_and_narrow(q) -> bool:
    """Whether a call's query is a plain contiguous tensor of a length and head dimension that the C++ autograd function takes: not
    decoding, and not head dimension 256, whose backward hands dS over."""
    return type(q) in _PLAIN and q.dim() == 4 and q.size(2) >= 128 and q.size(3) <= 128 and q.is_contiguous()


def ordinary(q, k, v) -> bool:
    """Whether a call whose query is `long_and_narrow` is one that the C++ autograd function serves exactly as the Python one does: plain
    contiguous tensors, outside function transforms, forward-mode differentiation, tracing, and modes that watch Python's calls."""
    return (type(k) in _PLAIN and type(v) in _PLAIN and k.is_contiguous() and v.is_contiguous()
            and torch._C._functorch.peek_interpreter_stack() is None and torch.autograd.forward_ad._current_level < 0
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0
            and torch._C._get_tracing_state() is None)


def attend(q, k, v, spec: MaskSpec, sm_scale, block_q, block_k, prepared):
    """o of a differentiable call without score function, bias and segment ids on `ordinary` tensors, or None where the call is not
    a prepared one or there is no C++ side.  ``prepared(q, k, v, spec)``: whether its shapes, mask and scale are (asked once per combination; it
    raises for what the entry points refuse)."""
    if q.dtype != k.dtype or q.dtype != v.dtype or k.shape != v.shape or q.device != k.device or q.device != v.device:
        return None   # (the general path says what is wrong)
    host = _lib.load_host()
    if host is None:
        return None
    key = (q.shape, k.shape, q.dtype, q.device, spec, sm_scale, block_q, block_k)
    plan = _attend_plans.get(key)
    if plan is False:
        return None
    maps = [ref() for ref in plan[1]] if plan is not None else (None,)
    if None in maps:
        if not prepared(q, k, v, spec):
            _attend_plans.put(key, False)
            return None
        parts = [_template(cls, pass_id, q, k, spec, sm_scale) for cls, pass_id in
                 ((_lib.FwdParamsC, _lib.PASS_FWD), (_lib.BwdParamsC, _lib.PASS_DQ), (_lib.BwdParamsC, _lib.PASS_DKV))]
        maps = [bm for _, bm in parts]
        plan = (host.Plan(*(t for t, _ in parts)), tuple(weakref.ref(bm) for bm in maps))
        _keep(_attend_plans, key, plan, maps)
    for bm in maps:   # (a map built on another stream: this one waits for it; the backward runs on this one too)
        bm.wait_ready(q.device)
    return host.attend(q, k, v, plan[0], maps[0].host_map(), maps[1].host_map(), maps[2].host_map())


def takes(q, k, spec: MaskSpec, sm_scale, *passes: int) -> bool:
    """Whether these passes of a checked call without score function and bias are prepared ones.  (Document ids keep arrays per stream,
    compiled masks their own libraries, and padded calls copy their operands: those go the general way.)"""
    _, _, Sq, D = q.shape
    Sk = k.shape[2]
    if spec.doc_ids is not None or spec.custom is not None or Sq < 128 or Sk < 128:
        return False
    if D == 128 or (D == 64 and q.dtype is torch.float32):   # (no question to the library in the usual cases)
        return True
    return all([call_head_dim(p, D, q.dtype, sm_scale, None, None, spec, Sq, Sk) == D for p in passes])


def forward(q, k, v, spec: MaskSpec, sm_scale, save_residuals, with_work=False):
    """(o, l, m), or o, of a call that `takes` accepts.  ``with_work``: through flexattn_fwd_work where that cuts
    the lists of a small grid (flex_attention's own forward)."""
    plan, maps = _plan((0, q.shape, k.shape, q.dtype, q.device, spec, sm_scale), q, k, spec, sm_scale, _lib.FwdParamsC, (_lib.PASS_FWD,))
    qp, kp, vp = q.data_ptr(), k.data_ptr(), v.data_ptr()
    if (qp | kp | vp) % 16:
        return forward(aligned(q), aligned(k), aligned(v), spec, sm_scale, save_residuals, with_work)
    o = torch.empty_like(q)
    l = m = None
    if save_residuals:
        l = torch.empty(q.shape[:3], dtype=torch.float32, device=q.device)
        m = torch.empty_like(l)
    p = _lib.FwdParamsC.from_buffer_copy(plan.templates[0])
    _FWD_POINTERS.pack_into(p, 0, qp, kp, vp, o.data_ptr(),
                            l.data_ptr() if save_residuals else 0, m.data_ptr() if save_residuals else 0)
    lib = _lib.load()
    with on_device(q.device):
        if with_work and plan.work_bytes is None:
            plan.work_bytes = lib.flexattn_fwd_work_bytes(C.byref(p))
        if with_work and plan.work_bytes > 0:
            work = torch.empty(plan.work_bytes, dtype=torch.uint8, device=q.device)
            _lib.check(lib.flexattn_fwd_work(C.byref(p), work.data_ptr(), plan.work_bytes, stream_of(q)), lib)
        else:
            _lib.check(lib.flexattn_fwd(C.byref(p), stream_of(q)), lib)
    return (o, l, m) if save_residuals else o


def backward(q, k, v, l, m, o, do, spec: MaskSpec, sm_scale):
    """(dq, dk, dv) of a call that `takes` accepts: delta, the dq and the dk/dv pass (flexattn_bwd)."""
    plan, maps = _plan((1, q.shape, k.shape, q.dtype, q.device, spec, sm_scale), q, k, spec, sm_scale, _lib.BwdParamsC,
                            (_lib.PASS_DQ, _lib.PASS_DKV))
    head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), do.data_ptr(), l.data_ptr(), m.data_ptr())
    op = o.data_ptr()
    if (head[0] | head[1] | head[2] | head[3] | op) % 16:
        return backward(aligned(q), aligned(k), aligned(v), l, m, aligned(o), aligned(do), spec, sm_scale)
    dq, dk, dv, delta = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.empty_like(l)
    pq = _lib.BwdParamsC.from_buffer_copy(plan.templates[0])
    pkv = _lib.BwdParamsC.from_buffer_copy(plan.templates[1])
    d = delta.data_ptr()
    _BWD_POINTERS.pack_into(pq, 0, *head, 0, dq.data_ptr(), 0, 0)
    _BWD_POINTERS.pack_into(pkv, 0, *head, d, 0, dk.data_ptr(), dv.data_ptr())
    pq.o, pq.delta_out = op, d
    lib = _lib.load()
    with on_device(q.device):
        _lib.check(lib.flexattn_bwd(C.byref(pq), C.byref(pkv), stream_of(q)), lib)
    return dq, dk, dv
