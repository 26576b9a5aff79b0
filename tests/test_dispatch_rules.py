"""The kernels' dispatch rules on the host: a driver compiled against csrc/q4d_internal.h asks the
library's own rule functions.  Nothing is launched."""

import subprocess
from pathlib import Path

import pytest

from llm_accelerator_amd import _lib

ROOT = Path(__file__).resolve().parents[1]
ROCM = Path("/opt/rocm")

DRIVER = r"""
#include <cstdio>
#include <cstring>
#include "q4d_internal.h"
using namespace q4d;
int main() {
  char rule[32];
  while (scanf("%31s", rule) == 1) {
    if (!strcmp(rule, "rows_tile")) {
      int M, N, K, count;
      if (scanf("%d %d %d %d", &M, &N, &K, &count) != 4) return 1;
      const RowsTile t = rows_tile(M, N, K, count);
      printf("%d %d %d\n", t.mt, t.nt, (int)t.k12);
    } else if (!strcmp(rule, "chain_resid")) {  // an output projection of a short prefill
      GemmArgs a;
      memset(&a, 0, sizeof(a));
      if (scanf("%d %d %d %d", &a.M, &a.N, &a.K, &a.ksplit) != 4) return 1;
      static float memory[64];  // aligned; never read
      a.nseg = 1;
      a.seg_end[0] = a.N;
      a.s[0] = (const uint16_t*)align_up((size_t)memory, 16);
      a.part = (float*)align_up((size_t)memory, 16);
      a.part_cap = (size_t)1 << 40;
      printf("%d\n", (int)chain_applies(a, EP_RESID, false));
    } else {
      return 1;
    }
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(DRIVER)
    subprocess.run([str(ROCM / "llvm/bin/clang++"), "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROOT / 'llm_accelerator_amd' / 'csrc'}", f"-I{ROCM / 'include'}", str(d / "rules.cpp"),
                    str(_lib.LIB_PATH), f"-Wl,-rpath,{_lib.LIB_PATH.parent}", f"-L{ROCM / 'lib'}",
                    f"-Wl,-rpath,{ROCM / 'lib'}", "-lamdhip64", "-o", str(d / "rules")], check=True)

    def ask(queries):
        """One list of numbers per query (rule name, arguments ...)."""
        text = "".join(" ".join(map(str, q)) + "\n" for q in queries)
        out = subprocess.run([str(d / "rules")], input=text, check=True, capture_output=True, text=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return ask


@pytest.mark.parametrize("count", [1, 2, 64])
@pytest.mark.parametrize("k", [1024, 2048, 3072])
def test_rows_tile_has_no_tile_of_padding_rows(rule, k, count):
    """Two row tiles a block only where there are two, whatever the matrix's width; a group keeps the
    waves that one matrix's launch has."""
    sizes = [(m, n) for m in (4, 16, 17, 32, 33, 500) for n in (2, 130, 3072, 12224, 12290, 40000, 151936)]
    tiles = rule([("rows_tile", m, n, k, count) for m, n in sizes])
    singles = rule([("rows_tile", m, n, k, 1) for m, n in sizes])
    assert len(tiles) == len(singles) == len(sizes)
    for (m, n), (mt, nt, k12), single in zip(sizes, tiles, singles):
        assert (mt, nt) in ((1, 1), (1, 2), (1, 4), (2, 4)) and 16 * (mt - 1) < m, (m, n)
        assert k12 == single[2] == (k == 3072 and single[:2] == [1, 1]), (m, n)
        if count > 1:
            assert mt == 1 or not k12
            assert nt in (1, 4), (m, n)   # the tiles that the grouped kernel has


def test_chain_resid_needs_a_split(rule):
    """The short prefill's output projections write raw partial tiles, which a reduction adds: without a
    split there is none, so y would never be written."""
    cases = [(m, n, k, ksplit) for m in (1, 75, 512) for n, k in ((1024, 512), (1024, 1024), (1024, 1536),
                                                                  (1024, 2048), (1024, 3072)) for ksplit in (0, 1, 2)]
    for c, (applies,) in zip(cases, rule([("chain_resid", *c) for c in cases])):
        assert applies == (c[3] == 2 and c[2] // 2 in (512, 1024, 1536)), c
