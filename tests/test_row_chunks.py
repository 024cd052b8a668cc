"""The addresses at which gemm_short.hip reads activation rows of any length (mindspore_amd/csrc/row_chunks.h, compiled for the host): every
chunk it fetches has a byte of the tensor in it, and every byte inside K that a lane takes out of LDS is its row's."""
import os
import shutil
import subprocess

import pytest

from mindspore_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include "mindspore_amd/csrc/row_chunks.h"

static void fail(const char *what, int m, int k, long base, int m0, int kb, int i) {
  printf("%s: m %d, k %d, address %ld, first row %d, K block %d, %d\n", what, m, k, base, m0, kb, i);
  exit(1);
}

static void walk(int m, int k, long base) {
  const long begin = base, behind = base + (long)m * k;
  for (int m0 = 0; m0 < m; m0 += 32) {
    const long tile = base + (long)m0 * k, from = tile - tile % 16;
    const mi::RowChunks c((uintptr_t)tile, m - m0, k);
    for (int kb = 0; kb < (k + 127) / 128; ++kb) {
      static long lds[5 * 64 * 16];
      for (int id = 0; id < 5 * 64; ++id) {
        const long at = from + c.of_block(c.first(id), kb);
        if (at % 16 != 0 || at + 16 <= begin || at >= behind) fail("chunk", m, k, base, m0, kb, id);
        for (int b = 0; b < 16; ++b) lds[id * 16 + b] = at + b;
      }
      for (int r = 0; r < 32 && m0 + r < m; ++r)
        for (int byte = 0; byte < 128 && kb * 128 + byte < k; ++byte)
          if (lds[r * 144 + c.odd(r) + byte] != base + (long)(m0 + r) * k + kb * 128 + byte) fail("byte", m, k, base, m0, kb, r);
    }
  }
}

int main() {
  const int ms[] = {1, 3, 32, 33, 64, 65, 97}, ks[] = {129, 130, 143, 144, 145, 255, 256, 257, 383, 1001, 2047};
  for (int m : ms)
    for (int k : ks)
      for (int odd = 0; odd < 16; ++odd) walk(m, k, 4096 + odd);
  const mi::RowChunks far((uintptr_t)4096, 1 << 20, 8000);  // (an end past 32 bits)
  if (far.of_block(far.first(287), 62) != 31 * 8000 + 128 + 62 * 128) fail("far", 1 << 20, 8000, 4096, 0, 62, 287);
  printf("ok\n");
  return 0;
}
"""


def test_row_chunks_have_bytes_of_the_tensor(tmp_path):
    src, exe = tmp_path / "chunks.cc", tmp_path / "chunks"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I" + ROOT, str(src), "-o", str(exe)])
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout


STRIDED = r"""
#include <stdio.h>
#include "gemm_core.h"

int main() {
  int8_t byte = 0;
  mi::GemmArgs g{};
  g.a = g.wb = &byte, g.c = &byte;
  g.m = 40, g.n = 64, g.k = 257, g.k_pad = 512, g.lda = 272, g.ldc = 64;
  for (int tile : {41, 81, 82})
    for (int requant = 0; requant < 2; ++requant) {
      const int rc = mi::launch_gemm_short(tile, true, requant != 0, false, g, mi::RequantParams{}, mi::DequantParams{}, nullptr);
      if (rc != MI_PARAM_INVALID) return printf("tile %d: status %d\n", tile, rc), 1;
    }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no compiler for the device's headers")
def test_rows_with_gaps_between_them_are_refused(tmp_path):
    """The chunks are those of rows end to end: others are refused before anything is launched."""
    src, exe = tmp_path / "strided.hip", tmp_path / "strided"
    src.write_text(STRIDED)
    subprocess.check_call(["hipcc", "--offload-host-only", "-std=c++17", "-I" + build.CSRC, str(src), "-o", str(exe), "-L" + build.HERE, "-lmi355x_int8",
                           "-Wl,-rpath," + build.HERE], stderr=subprocess.DEVNULL)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
