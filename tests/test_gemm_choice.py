"""The tiles that the GEMMs are tested on and those that they are run on: the choice (csrc/gemm_choice.h) is
plain C++, compiled here with the host compiler, and the shapes of the GPU tests have to reach every kernel
and tile that it can pick, for the served model's chunks and for the products of the op."""
import os
import shutil
import subprocess

import pytest

import qe
import test_gpu_chunk_gemm as chunks
import test_gpu_gemm_dma as products
from conftest import PKG

PROGRAM = r"""
#include <cstdio>
#include "gemm_choice.h"
using namespace qe;
int main() {
  char what;
  unsigned M, H, I, heads, kv;
  while (scanf(" %c", &what) == 1) {
    auto tile = [](const char* e, GemmTile t, unsigned depth) {
      printf("%s:%ux%u%s ", e, t.bm, t.bn, depth % 64 ? ":half" : "");
    };
    if (what == 'p') {  // a product M x N x K
      if (scanf("%u %u %u", &M, &H, &I) != 3) return 1;
      const GemmTile two = wide_pair_tile(M, H, I), s = kSliceTiles[slice_tile(M, H, I)];
      if (!gemm_on_wide(M, H, I)) printf("slice:%ux%u%s", s.bm, s.bn, s.bm == 16 && M <= 8 ? ":few" : "");
      else if (two.bn) tile("pair", two, I);
      else tile("wide", wide_tile(M, H, I, 1, false), I);
    } else {  // a chunk of M rows
      if (scanf("%u %u %u %u %u", &M, &H, &I, &heads, &kv) != 5) return 1;
      if (chunk_on_split_rows(M, H, I)) {
        tile("qkv", wide_tile(M, (heads + 2 * kv) * 128, H, 1, true), H);
        for (unsigned K : {heads * 128, I}) {
          const unsigned z = gemm_splits(M, H, K);
          tile("partial", wide_tile(M, H, K / z, z, false), K / z);
        }
        tile("silu", wide_tile(M, 2 * I, H, 1, false), H);
      } else {
        printf("rows");
      }
    }
    printf("\n");
  }
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    """lines of questions -> the answers, one set of words each"""
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("choice")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(PKG, "csrc"), "-o",
                    str(d / "choose"), str(d / "main.cpp")], check=True)

    def ask(lines):
        out = subprocess.run([str(d / "choose")], input="\n".join(lines), capture_output=True, text=True, check=True)
        return [set(line.split()) for line in out.stdout.splitlines()]

    return ask


def chunk_line(c, m):
    return f"c {m} {c.hidden_size} {c.intermediate_size} {c.num_attention_heads} {c.num_key_value_heads}"


def test_chunks_of_the_served_model_run_on_tested_tiles(choose):
    tested = set().union(*choose([chunk_line(chunks.CONFIGS[name], n) for name, n, _ in chunks.CASES]))
    served = set().union(*choose([chunk_line(qe.QWEN3_0_6B, m) for m in range(65, 2049)]))
    assert served <= tested, f"no test reaches {sorted(served - tested)}"
    # widths that are no multiple of 64, on both sides of their own limit
    other = [qe.Config(1056, 3104, 1, 16, 8, 128, 1000, 1e-6, 1e6, 999),
             qe.Config(2080, 4064, 1, 16, 8, 128, 1000, 1e-6, 1e6, 999)]
    half = set().union(*choose([chunk_line(c, m) for c in other for m in range(65, 2049)]))
    assert "rows" in half and half <= tested, f"no test reaches {sorted(half - tested)}"


def test_products_run_on_tested_tiles(choose):
    tested = set().union(*choose([f"p {m} {n} {k}" for m, n, k in products.SHAPES]))
    ms = sorted({int(2 * 1.11 ** i) for i in range(67)} | {8, 9, 64, 65, 2048})
    nks = [(n, k) for n in (2, 128, 512, 1022, 1024, 2526, 4096, 5110, 6144, 16384, 151936)
           for k in (32, 64, 96, 320, 512, 544, 1024, 1056, 2048, 3072)]
    run = set().union(*choose([f"p {m} {n} {k}" for m in ms for n, k in nks]))
    assert run <= tested, f"no test reaches {sorted(run - tested)}"
