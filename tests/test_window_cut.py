"""Which convolutions keep a second copy of their weights for the windows in LDS (mindspore_amd/csrc/window_cut.h, compiled for the host):
those for which images exist that run on it, only those, and but for a few oddities all."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <random>
#include "mindspore_amd/csrc/window_cut.h"

using mi::ConvGeom;

static std::mt19937 rng(1);
static int draw(int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); }

static void fail(const char *what, const ConvGeom &g) {
  printf("%s: %d x %d x %d x %d -> %d x %d x %d, taps %d x %d, strides %d %d, dilations %d %d\n", what, g.batch, g.in_h, g.in_w, g.in_c, g.out_h,
         g.out_w, g.out_c, g.kernel_h, g.kernel_w, g.stride_h, g.stride_w, g.dilation_h, g.dilation_w);
  exit(1);
}

static ConvGeom of_output(ConvGeom g, int batch, int out_h, int out_w) {
  g.batch = batch, g.out_h = out_h, g.out_w = out_w;
  g.in_h = (out_h - 1) * g.stride_h + (g.kernel_h - 1) * g.dilation_h + 1;
  g.in_w = (out_w - 1) * g.stride_w + (g.kernel_w - 1) * g.dilation_w + 1;
  return g;
}

// some image runs on it: the smallest that can, or one of those drawn
static bool some_image(const ConvGeom &g, bool *small) {
  mi::WindowCut c;
  *small = false;
  for (int w = 8; w <= 64 && !*small; ++w)
    for (int h = (127 + w) / w; h <= 256 / w && !*small; ++h)
      for (int batch : {168, 256, 512, 768, 2048}) *small = *small || mi::choose_window(of_output(g, batch, h, w), true, &c);
  if (*small) return true;
  for (int i = 0; i < 200; ++i)
    if (mi::choose_window(of_output(g, draw(1, 600), draw(1, 120), draw(1, 120)), true, &c)) return true;
  return false;
}

static ConvGeom geometry(int in_c, int out_c, int taps, int stride) {
  return ConvGeom{1, 16, 16, in_c, 1, 1, out_c, taps, taps, stride, stride, 1, 1, 0, 0};
}

int main() {
  if (mi::window_fits(geometry(128, 128, 3, 1))) fail("weights that no image runs on", geometry(128, 128, 3, 1));
  if (mi::window_fits(geometry(128, 97, 3, 2))) fail("weights that no image runs on", geometry(128, 97, 3, 2));
  if (!mi::window_fits(geometry(64, 64, 3, 1))) fail("none", geometry(64, 64, 3, 1));
  if (!mi::window_fits(geometry(64, 128, 3, 2))) fail("none", geometry(64, 128, 3, 2));
  if (!mi::window_fits(geometry(128, 96, 3, 1))) fail("none", geometry(128, 96, 3, 1));
  if (!mi::window_fits(geometry(3, 96, 7, 2))) fail("none", geometry(3, 96, 7, 2));
  int seen[2] = {}, odd = 0;
  for (int i = 0; i < 4000; ++i) {
    ConvGeom g = geometry(draw(0, 3) == 0 ? draw(3, 4) : 16 * draw(1, 16), draw(1, 130), 1, 1);
    g.kernel_h = draw(1, 8), g.kernel_w = draw(1, 8), g.stride_h = draw(1, 4), g.stride_w = draw(1, 4);
    g.dilation_h = draw(1, 3), g.dilation_w = g.in_c <= 4 ? 1 : draw(1, 3);
    bool small;
    const bool some = some_image(g, &small), fits = mi::window_fits(g);
    if (some && !fits) ++odd;  // (some number of rectangles just fills their rounds and not the GEMM's)
    if (fits && !small) fail("weights that no image runs on", g);
    ++seen[fits];
  }
  if (seen[0] < 200 || seen[1] < 200 || odd > 40) return printf("kept %d, not kept %d, of which with images %d\n", seen[1], seen[0], odd), 1;
  printf("ok\n");
  return 0;
}
"""


def test_window_weights_are_kept_where_images_run_on_them(tmp_path):
    src, exe = tmp_path / "cut.cc", tmp_path / "cut"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-I" + ROOT, str(src), "-o", str(exe)])
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout
