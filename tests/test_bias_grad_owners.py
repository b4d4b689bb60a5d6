"""Ragged lengths start their last tile early, so two work-groups of the dk/dv pass compute the elements both tiles hold.
Which of them stores the bias gradient of an element (fa::tile_base and fa::first_owned in fa_common.hpp, from their C++
text): exactly one, for every element, lane and row block as the kernel walks them."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flex_attention_tpu_amd", "csrc")
WALK = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
int main(int argc, char** argv) {
  const int Sq = atoi(argv[1]), Sk = atoi(argv[2]), T = 128;
  const int nq = (Sq + T - 1) / T, nk = (Sk + T - 1) / T;
  std::vector<unsigned char> n((size_t)Sq * Sk, 0);
  for (int kb = 0; kb < nk; ++kb)
    for (int kv = 0; kv < T; ++kv) {
      const int k_idx = tile_base(kb, T, Sk) + kv;
      const bool own_col = k_idx >= kb * T;
      for (int qb = 0; qb < nq; ++qb) {
        const int q0 = tile_base(qb, T, Sq);
        // (a tile cut off at Sk is at most partial, a last q tile that starts early counts as partial)
        const bool masked = (kb + 1) * T > Sk || (qb + 1) * T > Sq;
        for (int hh = 0; hh < 2; ++hh) {
          const int own = first_owned(qb, T, q0, 4 * hh, own_col);
          for (int r = 0; r < 16; ++r)       // (lane half hh: rows 8 r + 4 hh + 0..3 of the tile)
            for (int u = 0; u < 4; ++u)
              if (!masked || 8 * r + u >= own) ++n[(size_t)(q0 + 8 * r + 4 * hh + u) * Sk + k_idx];
        }
      }
    }
  for (size_t i = 0; i < n.size(); ++i)
    if (n[i] != 1) { printf("row %d column %d: %d stores\n", (int)(i / Sk), (int)(i % Sk), n[i]); return 1; }
  return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    text = open(os.path.join(CSRC, "fa_common.hpp")).read()
    fns = [re.search(r"__host__ __device__ __forceinline__ (int %s\(.*?\n\})" % name, text, re.S).group(1) for name in ("tile_base", "first_owned")]
    d = tmp_path_factory.mktemp("owners")
    (d / "w.cpp").write_text("\n".join(fns) + WALK)
    subprocess.check_call(["g++", "-O1", "-o", str(d / "w"), str(d / "w.cpp")])
    return str(d / "w")


@pytest.mark.parametrize("Sq,Sk", [(128, 128), (128, 129), (129, 128), (191, 257), (255, 385), (1500, 1500), (640, 321)])
def test_every_element_has_one_writer(walk, Sq, Sk):
    r = subprocess.run([walk, str(Sq), str(Sk)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_the_kernel_stores_what_it_owns():
    text = open(os.path.join(CSRC, "bwd_dkv_bf16.hip")).read()
    stores = [line for line in text.splitlines() if "raw_buffer_store" in line]
    assert len(stores) == 1 and "if (DAB)" in stores[0] and "dab_off" in stores[0]
    assert "const bool owned = 32 * cc + 8 * g4 + u >= own;" in text and "dab_off = owned ? dab_off : ~0u;" in text
