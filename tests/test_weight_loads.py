"""The byte ranges of the packed weights that the K-block GEMM loops ask for (mindspore_amd/csrc/weight_loads.h, compiled for
the host): every loader instruction of every wave, tile shape and K block lies inside the packed weights, and the groups that
exist are loaded from their own place."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include "mindspore_amd/csrc/weight_loads.h"

static const int kPad = 256;  // kNPad, kKPad
static long checked = 0;

static void fail(const char *what, int tn, int n, int k, int n0, int wave, int i, int kb) {
  printf("%s: TN %d, n %d, k %d, n0 %d, wave %d, instruction %d, K block %d\n", what, tn, n, k, n0, wave, i, kb);
  exit(1);
}

template <int TN>
static void tile(int n, int k) {
  const int n_pad = (n + kPad - 1) / kPad * kPad, k_pad = (k + kPad - 1) / kPad * kPad;
  const int ldw = (k_pad / 256) % 2 == 0 ? k_pad + 256 : k_pad, k64 = k_pad / 64, kblocks = (k + 127) / 128;
  const int64_t blocked = (int64_t)n_pad * k_pad, rows = (int64_t)n_pad * ldw;
  for (int n0 = 0; n0 < n; n0 += 64 * TN)
    for (int wave = 0; wave < 4; ++wave) {
      const mi::WaveWeightGroups<TN> wg(n, n0, wave, kPad);
      const int own = n0 / 16 + wave * TN;
      if (wg.inside < 1 || wg.inside > TN) fail("no group", TN, n, k, n0, wave, -1, -1);
      for (int i = 0; i < 2 * TN; ++i) {
        const int group = wg.first + wg.group(i >> 1);
        if (group < 0 || group >= n_pad / 16) fail("group", TN, n, k, n0, wave, i, -1);
        if (own + (i >> 1) < n_pad / 16 && group != own + (i >> 1)) fail("another group", TN, n, k, n0, wave, i, -1);
        for (int kb = 0; kb < kblocks; ++kb) {
          const int64_t b = (int64_t)wg.first * k64 * 1024 + mi::blocked_weight_offset(wg.group(i >> 1), i & 1, k64, kb);
          if (b < 0 || b + 1024 > blocked) fail("blocked", TN, n, k, n0, wave, i, kb);
          if (b != ((int64_t)group * k64 + 2 * kb + (i & 1)) * 1024) fail("blocked place", TN, n, k, n0, wave, i, kb);
          const int64_t r = (int64_t)wg.first * 16 * ldw + mi::row_major_weight_offset(wg.group(i >> 1), i & 1, ldw, kb);
          if (r < 0 || r + 7 * ldw + 128 > rows) fail("row-major", TN, n, k, n0, wave, i, kb);
          if (r != ((int64_t)group * 16 + 8 * (i & 1)) * ldw + 128 * kb) fail("row-major place", TN, n, k, n0, wave, i, kb);
          ++checked;
        }
      }
    }
}

int main() {
  const int ks[] = {16, 128, 144, 256, 272, 1040, 4096};
  for (int k : ks)
    for (int n = 1; n < 2400; n += n < 800 ? 1 : 37) {
      tile<1>(n, k);
      tile<2>(n, k);
      tile<3>(n, k);
      tile<4>(n, k);
    }
  tile<3>(11008, 4096);
  tile<3>(9003, 1040);
  tile<3>(65536 + 5, 8192);
  printf("%ld ok\n", checked);
  return 0;
}
"""


def test_weight_loads_stay_inside_the_packed_weights(tmp_path):
    src, exe = tmp_path / "loads.cc", tmp_path / "loads"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I" + ROOT, str(src), "-o", str(exe)])
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0 and p.stdout.endswith(" ok\n"), p.stdout
