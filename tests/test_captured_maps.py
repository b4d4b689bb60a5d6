"""Block maps of calls that are captured into a graph: built when the graph is replayed and not before, so no call outside of that
capture may be handed one, through whichever cache.  On the CPU: the builder, the streams and the launches are stand-ins, the caches
and the plans are the package's own."""
import contextlib
import types

import pytest
import torch

from flex_attention_tpu_amd import _lib, _plans, block_mask
from flex_attention_tpu_amd.masks import MaskSpec


class _Event:
    def record(self, stream):
        pass


class _Gpu:
    """What stands in for the device: which capture the current stream is part of (0: none), and the launches."""

    def __init__(self):
        self.capture, self.built, self.launched = 0, [], []
        self.stream = types.SimpleNamespace(cuda_stream=7, wait_event=lambda event: None)

    def build(self, *args):
        self.built.append(self.capture)
        return 0

    def attend(self, q, k, v, plan, *maps):
        self.launched.append(maps)
        return q


@pytest.fixture
def gpu(monkeypatch):
    gpu = _Gpu()
    lib = _lib.load()
    monkeypatch.setattr(_lib, "load_for", lambda *a: types.SimpleNamespace(flexattn_build_block_mask_ragged=gpu.build))
    monkeypatch.setattr(_lib, "load_host", lambda: types.SimpleNamespace(Plan=lambda *a: a, Map=lambda *a: a, attend=gpu.attend))
    monkeypatch.setattr(lib, "flexattn_last_error_string", lambda: b"")
    monkeypatch.setattr(block_mask, "raw_stream", lambda device: 7)
    monkeypatch.setattr(block_mask, "_capturing", lambda: gpu.capture != 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: gpu.stream)
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    for module, name in ((block_mask, "_map_cache"), (_plans, "_plans"), (_plans, "_attend_plans")):
        monkeypatch.setattr(module, name, block_mask.LRU(64))
    return gpu


def attend(q, k, v):
    return _plans.attend(q, k, v, MaskSpec(_lib.MASK_CAUSAL), 0.1, 128, 128, lambda *a: True)


def prepared(q, k, v):
    return _plans._plan((0, q.shape), q, k, MaskSpec(_lib.MASK_CAUSAL), 0.1, _lib.FwdParamsC, (_lib.PASS_FWD,))[1]


def general(q, k, v):
    return [block_mask.build_block_map(MaskSpec(_lib.MASK_CAUSAL), 256, 256, 128, 128, q.device)]


@pytest.mark.parametrize("call", [attend, prepared, general])
@pytest.mark.parametrize("order", [(1, 0, 2, 0), (1, 2, 0), (0, 1, 0)])
def test_no_call_is_handed_a_map_of_another_capture(gpu, order, call):
    """Calls of one combination inside (1, 2) and outside (0) of captures: a map that an eager call built serves all that follow,
    one that a captured call built that capture alone."""
    q, k, v = (torch.empty(1, 2, 256, 128, dtype=torch.bfloat16) for _ in range(3))
    born = []   # (map, capture that built it)
    for n, capture in enumerate(order):
        gpu.capture, before = capture, len(gpu.built)
        out = call(q, k, v)
        for used in gpu.launched[-1] if call is attend else out:
            if not any(m is used for m, _ in born):
                born.append((used, capture))
            assert all(c in (0, capture) for m, c in born if m is used)
        assert set(gpu.built[before:]) == (set() if 0 in order[:n] else {capture})
