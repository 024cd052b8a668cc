"""The byte ranges of the packed weights that the K-block GEMM loops ask for (mindspore_amd/csrc/weight_loads.h, compiled for
the host): every loader instruction of every wave, tile shape and K block lies inside the packed weights, and the groups that
exist are loaded from their own place."""
import os
import shutil
import subprocess

import pytest

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


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no compiler for the device")
def test_no_load_goes_round_a_loop_over_descriptors(tmp_path):
    """The K-block loops' loads are given descriptors and offsets that are the same in every lane.  Where the compiler does not see
    that, it puts each load into a loop over the lanes' values (row-major weights, 2048 x 2048 x 2048 with weight zero points
    13.2 -> 15.9 us): a load under a narrowed exec mask, and a branch back while there are lanes left."""
    from mindspore_amd import build
    text = open(os.path.join(build.CSRC, "gemm_kblock.hip")).read()
    kernels = text[:text.index("template <int TN, int TM, int EPI, bool HAS_ZW, bool FAST>\nstatic int launch_kblock(")]  # without the host's choice among all
    src, asm = tmp_path / "kblock.hip", tmp_path / "kblock.s"
    src.write_text(kernels + "".join("template __global__ void gemm_kblock_kernel<%s>(GemmCall<%s>);\n" % (form, form.split(",")[2]) for form in
                                     ("2, 2, 0, true, true, false", "2, 2, 1, false, true, false", "2, 2, 0, false, true, true")) + "}\n")
    subprocess.check_call(["hipcc"] + build.FLAGS + ["-I" + build.CSRC, "--cuda-device-only", "-S", str(src), "-o", str(asm)],
                          stderr=subprocess.DEVNULL)
    lines = [s.split(";")[0].split() for s in asm.read_text().splitlines()]
    lines = [s for s in lines if s and (s[0].startswith(("s_", "buffer_")) or s[0].endswith(":"))]
    loads = [i for i, s in enumerate(lines) if s[0].startswith("buffer_load") and s[-1] == "lds"]
    assert len(loads) >= 60  # (they were found)
    assert not [lines[i] for i in loads if lines[i + 1][0] == "s_xor_b64" and lines[i + 1][1] == "exec," and lines[i + 2][0] == "s_cbranch_execnz"]
