"""Block maps of calls that are captured into a graph: built when the graph is replayed and not before, so no call outside of that
capture may be handed one, through whichever cache.  On the CPU: the builder, the streams and the launches are stand-ins, the caches
and the plans are the package's own."""
import contextlib
import gc
import types
import weakref

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
        self.capture, self.built, self.launched, self.ended = 0, [], [], []
        self.stream = types.SimpleNamespace(cuda_stream=7, wait_event=lambda event: None)

    def build(self, *args):
        self.built.append(self.capture)
        return 0

    def captures_ended(self, tokens, n):
        some, self.ended = self.ended[:n], self.ended[n:]
        tokens[:len(some)] = some
        return len(some)

    def attend(self, q, k, v, plan, *maps):
        self.launched.append(maps)
        return q


@pytest.fixture
def gpu(monkeypatch):
    gpu = _Gpu()
    lib = _lib.load()
    monkeypatch.setattr(_lib, "load_for", lambda *a: types.SimpleNamespace(flexattn_build_block_mask_ragged=gpu.build))
    monkeypatch.setattr(_lib, "load_host", lambda: types.SimpleNamespace(Plan=lambda *a: a, Map=lambda *a: a, attend=gpu.attend))
    monkeypatch.setattr(lib, "flexattn_capture_token", lambda stream: gpu.capture)
    monkeypatch.setattr(lib, "flexattn_captures_ended", gpu.captures_ended)
    monkeypatch.setattr(block_mask, "raw_stream", lambda device: 7)
    monkeypatch.setattr(block_mask, "_capturing", lambda: gpu.capture != 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: gpu.stream)
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    for module, name in ((block_mask, "_map_cache"), (_plans, "_plans"), (_plans, "_attend_plans")):
        monkeypatch.setattr(module, name, block_mask.LRU(64))
    yield gpu
    gpu.capture, gpu.ended = 0, list(range(1, 400))
    block_mask.release_ended()


def attend(q, k, v):
    return _plans.attend(q, k, v, MaskSpec(_lib.MASK_CAUSAL), 0.1, 128, 128, lambda *a: True)


def prepared(q, k, v):
    return _plans._plan((0, q.shape, k.shape), q, k, MaskSpec(_lib.MASK_CAUSAL), 0.1, _lib.FwdParamsC, (_lib.PASS_FWD,))[1]


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


@pytest.mark.parametrize("known", [True, False])
def test_a_graph_s_maps_live_as_long_as_it(gpu, known):
    """However many other captures there are, and no longer: known maps (that an eager call built and the cache then drops) and maps
    of the capture's own."""
    graphs = {}   # capture -> what its calls read
    for n in range(1, 400):
        q, k, v = (torch.empty(1, 2, 128 * m, 128, dtype=torch.bfloat16) for m in (n % 20 + 1, n // 20 + 1, n // 20 + 1))
        if known:
            gpu.capture = 0
            prepared(q, k, v)
        gpu.capture = n
        graphs[n] = [weakref.ref(bm) for bm in prepared(q, k, v)]
        gpu.capture = 0
        block_mask._map_cache.clear()
    gc.collect()
    assert all(ref() is not None for refs in graphs.values() for ref in refs)
    gpu.ended = [n for n in graphs if n % 2]
    general(q, k, v)   # (any call that builds a map looks for ended graphs)
    block_mask._map_cache.clear()
    gc.collect()
    assert all((ref() is None) == (n % 2 == 1) for n, refs in graphs.items() for ref in refs)


def test_one_capture_builds_a_map_once(gpu):
    """The calls of a capture share the maps that it builds, as eager calls share theirs."""
    q, k, v = (torch.empty(1, 2, 256, 128, dtype=torch.bfloat16) for _ in range(3))
    for gpu.capture in (1, 2):
        before = len(gpu.built)
        for call in (attend, prepared, general):
            call(q, k, v)
            if call is attend:
                first = len(gpu.built)
        assert before < first and len(gpu.built) <= first + 1   # (general: a map at blocks of its own)


def test_a_graph_s_ids_and_slopes_live_as_long_as_it(gpu, monkeypatch):
    """The other arrays that parameter blocks point at and that bounded caches hold: document ids, their ranges, position-bias
    slopes."""
    from flex_attention_tpu_amd import _common
    from flex_attention_tpu_amd.masks import DocIds
    from flex_attention_tpu_amd.scores import make_alibi_global_score_fn
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, stream: None)
    caches = [(block_mask, "_doc_cache"), (block_mask, "_range_cache"), (block_mask, "_rows_cache"), (_common, "_slopes_cache")]
    for module, name in caches:
        monkeypatch.setattr(module, name, block_mask.LRU(64))
    cpu = torch.device("cpu")
    shared, entries = torch.arange(256) // 100, torch.stack([torch.arange(256) // n for n in (60, 90)])
    specs = [MaskSpec(_lib.MASK_DOC, doc_ids=DocIds(ids.numpy())) for ids in (shared, entries)]

    def call():
        for spec in specs:
            block_mask.mask_spec_c(spec, 256, 256, cpu)
        _common.score_spec_c(make_alibi_global_score_fn(4), 4, cpu, 128, 128)
    call()   # (a captured call copies nothing to the device: the arrays are an eager call's)
    gpu.capture = 1
    call()
    gpu.capture = 0
    arrays = [weakref.ref(t) for module, name in caches for t in getattr(module, name)._d.values() if isinstance(t, torch.Tensor)]
    assert len(arrays) >= 4
    for module, name in caches:
        getattr(module, name).clear()
    gc.collect()
    assert all(ref() is not None for ref in arrays)
    gpu.ended = [1]
    block_mask.release_ended()
    gc.collect()
    assert all(ref() is None for ref in arrays)
