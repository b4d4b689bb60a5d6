"""The host side of the block maps' caches."""
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
