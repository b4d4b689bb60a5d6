"""The host side of the block maps' caches."""
import collections
import sys
import threading

import pytest

from flex_attention_tpu_amd import block_mask
from flex_attention_tpu_amd.masks import MaskSpec


def test_ragged_lengths_are_refused_whether_cached_or_not(monkeypatch):
    """create_block_mask takes whole blocks only, also once an attention call has left the ragged map in the cache."""
    cache = block_mask.LRU(4)
    monkeypatch.setattr(block_mask, "_map_cache", cache)
    for cached in (False, True):
        if cached:
            cache.put((MaskSpec(), 200, 256, 128, 128, "cuda"), object())
        with pytest.raises(ValueError, match="divisible"):
            block_mask.create_block_mask(MaskSpec(), 200, 256, 128, 128)


def test_lru_shared_by_threads():
    """Threads that look up, add and drop entries of one small cache at once: no lookup and no addition raises, and the
    bound holds."""
    lru, errors, interval = block_mask.LRU(2), [], sys.getswitchinterval()

    def work(seed):
        try:
            for i in range(20000):
                k = (seed * 7 + i * 3) % 5
                if lru.get(k) is None:
                    lru.put(k, object())
                if i % 500 == 0:
                    lru.clear()
        except Exception as e:   # (reported by the test's own thread)
            errors.append(e)
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(s,)) for s in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not errors, errors[:3]
    assert len(lru) <= 2


def test_lru_entry_dropped_while_it_is_added():
    """Another thread fills the cache right behind an addition's first step: the addition still ends without an error."""
    lru = block_mask.LRU(1)

    class Interrupted(collections.OrderedDict):
        def __setitem__(self, key, value):
            super().__setitem__(key, value)
            if key == "a":
                other.start()
                other.join(0.3)   # (done by then, or waiting for this addition)
    other = threading.Thread(target=lambda: (lru.put("b", 1), lru.put("c", 1)))
    lru._d = Interrupted()
    lru.put("a", 1)
    other.join()
    assert len(lru) == 1
