"""The order in which work-groups that take one item each start (fa::single_item in fa_common.hpp), from its C++ text: every
(head, block) once, each XCD's heads a contiguous share, and within a set of heads the blocks of equal rank together."""
import os
import re

import pytest

HPP = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flex_attention_tpu_amd", "csrc", "fa_common.hpp")


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    import ctypes
    import subprocess
    text = open(HPP).read()
    body = re.search(r"constexpr int kSetItems = \d+;\n__host__ __device__ (inline void single_item.*?\n\})", text, re.S)
    n = re.search(r"constexpr int kSetItems = \d+;", text).group(0)
    d = tmp_path_factory.mktemp("single_item")
    (d / "s.cpp").write_text(n + "\n" + body.group(1) + '\nextern "C" void item(int j, int n, int nb, int* h, int* k) { single_item(j, n, nb, *h, *k); }\n')
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", "-o", str(d / "s.so"), str(d / "s.cpp")])
    lib = ctypes.CDLL(str(d / "s.so"))

    def item(j, n_wg, nb):
        h, k = ctypes.c_int(), ctypes.c_int()
        lib.item(j, n_wg, nb, ctypes.byref(h), ctypes.byref(k))
        return h.value, k.value
    return item


@pytest.mark.parametrize("heads", [1, 3, 8, 12, 16, 24, 40, 64, 256])
@pytest.mark.parametrize("blocks", [1, 2, 5, 11, 16, 63, 64, 100])
def test_every_item_once(order, heads, blocks):
    n = heads * blocks
    items = [order(j, n, blocks) for j in range(n)]
    assert sorted(items) == [(h, k) for h in range(heads) for k in range(blocks)]
    if heads % 8 == 0:
        for x in range(8):
            mine = items[x::8]
            assert {h for h, _ in mine} == set(range(x * heads // 8, (x + 1) * heads // 8))
            together = max(1, 64 // blocks)      # heads of a set
            for first in range(0, heads // 8, together):
                ranks = [k for h, k in mine if first <= h - x * heads // 8 < first + together]
                assert ranks == sorted(ranks)
