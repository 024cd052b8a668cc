"""The addresses at which gemm_short.hip reads activation rows of any length (mindspore_amd/csrc/row_chunks.h, compiled for the host): every
chunk it fetches has a byte of the tensor in it, and every byte inside K that a lane takes out of LDS is its row's."""
import os
import subprocess

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
