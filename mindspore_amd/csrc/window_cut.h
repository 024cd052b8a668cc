// Which convolutions run with their window's pixels in LDS (conv_window.hip), and in which rectangles.  Plain integer arithmetic, walked on
// the host by tests/test_window_cut.py.
#pragma once

#include <stdint.h>

#include <algorithm>

#include "conv_geom.h"

namespace mi {

constexpr int kWaves = 8;  // of a workgroup, 32 output pixels each
// Blocks of 32 channels that a workgroup computes.
static inline int window_blocks(const ConvGeom &g) { return (g.out_c + 31) / 32; }

// few channels, four bytes a pixel in LDS
static inline bool packed_window(const ConvGeom &g) { return g.in_c <= 4; }
static inline int row_chunks(const ConvGeom &g) { return (g.kernel_w + 3) / 4; }

constexpr int kWindowLds = 80 << 10;  // two workgroups per CU
constexpr int kWindowLdsWide = 160 << 10;  // one, of more than 64 channels
struct WindowCut {
  int tile_h, tile_w, tiles_x, tiles_y, patch_h, patch_w, pitch, steps, weight_bytes, patch_bytes;
  int64_t tiles;
};
static inline int window_lds(const ConvGeom &g) { return window_blocks(g) > 2 && !packed_window(g) ? kWindowLdsWide : kWindowLds; }
// The rectangles of an image that need the fewest workgroups, and of those the fewest input pixels; false if none fits.
static inline bool cut_window(const ConvGeom &g, WindowCut *best) {
  const int cc = g.in_c / 16, most = 32 * kWaves;  // (tile_w <= most)
  WindowCut c{};
  const bool packed = packed_window(g);
  c.pitch = cc | 1;
  c.steps = packed ? (g.kernel_h * row_chunks(g) + 1) / 2 : (g.kernel_h * g.kernel_w * cc + 1) / 2;
  c.weight_bytes = window_blocks(g) * c.steps * 1024;
  best->tiles = 0;
  for (int nx = (g.out_w + 63) / 64, last = std::min(64, (g.out_w + 7) / 8); nx <= last; ++nx) {  // 8 to 64 pixels wide
    c.tile_w = (g.out_w + nx - 1) / nx;
    if (c.tile_w < 8) continue;
    c.tiles_x = (g.out_w + c.tile_w - 1) / c.tile_w;
    c.tile_h = std::min(most / c.tile_w, g.out_h);
    c.tiles_y = (g.out_h + c.tile_h - 1) / c.tile_h;
    c.tile_h = (g.out_h + c.tiles_y - 1) / c.tiles_y;
    const int64_t ph = (int64_t)(c.tile_h - 1) * g.stride_h + (int64_t)(g.kernel_h - 1) * g.dilation_h + 1;
    int64_t pw = (int64_t)(c.tile_w - 1) * g.stride_w +
                 (packed ? 4 * row_chunks(g) : (int64_t)(g.kernel_w - 1) * g.dilation_w + 1);
    if (packed) pw = (pw + 3) & ~3;
    if (ph > 4096 || pw > 4096) continue;
    c.patch_h = (int)ph;
    c.patch_w = (int)pw;
    const int64_t patch = (ph + (packed ? g.dilation_h : 0)) * pw * (packed ? 4 : c.pitch * 16);
    const int64_t bytes = (patch + 1023) / 1024 * 1024;  // (at most kWindowLdsWide, hence fewer than 2^16 chunks)
    if (c.weight_bytes + bytes + 8 * c.steps > window_lds(g)) continue;
    c.patch_bytes = (int)bytes;
    c.tiles = (int64_t)c.tiles_x * c.tiles_y * g.batch;
    const bool fewer = c.tiles < best->tiles || (c.tiles == best->tiles && c.patch_bytes < best->patch_bytes);
    if (best->tiles == 0 || fewer) *best = c;
  }
  return best->tiles != 0;
}

// Up to 128 channels, which one workgroup computes (more would fetch the pixels again), rectangles for two CUs in three, and at
// least half of their pixels there.  Time of this relative to the gathering GEMM, 3x3: workgroups 112 1.01, 128 1.02, 140 1.02,
// 160 1.02, 168 0.88 0.91, 192 0.87, 196 0.89, 224 0.87, 256 0.77, 448 0.75, 1024 0.70; stride 2 256 0.74; 5x5 128 0.84, 256 0.73.
// Rectangles filled to 0.77 0.77, 0.56 0.87, 0.39 0.90 to 1.05, 0.25 1.43, 0.19 1.40 to 2.1.
// 65 to 96 channels, of which the GEMM's 128-channel tiles leave a quarter and more empty, already from 96 workgroups: 96 -> 96 56 1.02,
// 98 0.84, 112 0.86, 224 0.72, 448 0.66, 64 -> 96 56 1.10, 112 0.90, 448 0.61, 32 -> 72 896 0.55; 97 to 128: 64 -> 128 112 1.03, 128 1.04,
// 224 0.84, 448 0.82, 32 -> 128 252 0.89.
// Three or four channels: windows for which conv_rows_kernel makes five or more loads.  Time relative to that one, us: 7x7 on 3
// channels -> 64, 49 workgroups 4.42 / 4.42, 98 4.46 / 4.48, 196 6.2 / 4.65, 392 8.55 / 6.05, 784 12.2 / 9.55, 1568 20.5 / 16.5;
// -> 96, 49 4.82 / 4.89, 98 6.71 / 5.06, 1568 35.9 / 19.6, -> 128, 98 6.78 / 5.73, 1568 38.1 / 24.0;
// 5x5 on 4 (five loads) 4.85 / 4.4 and 14.8 / 14.7, -> 96, 90 workgroups 5.10 / 4.55; 5x5 on 3 (three) 4.15 / 4.18; 3x3 on 3 (two)
// 5.17 / 5.55 and 7.7 / 8.8.
constexpr int kWindowLeastTiles = 168, kWindowLeastWideTiles = 96;
static inline int least_tiles(const ConvGeom &g) {
  return window_blocks(g) == 3 || (window_blocks(g) == 4 && packed_window(g)) ? kWindowLeastWideTiles : kWindowLeastTiles;
}
// More than 64 channels beside several taps of 16-channel-aligned images mostly leave room for one workgroup a CU, and what counts then is
// how many rounds of them there are beside those of the GEMM's 128 x 128 tiles, two a CU.  A round takes 0.7 of one of those for 65 to 96
// channels, 0.85 to 0.9 for up to 128 (full rounds: 96 -> 96 8.75 / 12.5, 64 -> 128 7.85 / 9.35); two a CU as long as one of the GEMM's
// rounds and do twice as much.  Relative time at 252 workgroups (against one of the GEMM's rounds) 0.70, 266 1.11, 280 1.18 (not taken),
// 336 (against two) 0.78, 512 0.69, 518 0.95 (not taken); 64 -> 128 336 0.96, 518 1.14 (not taken).
static inline bool wide_rounds_pay(const ConvGeom &g, const WindowCut &c) {
  if (window_blocks(g) < 3 || packed_window(g)) return true;
  const bool two = window_blocks(g) == 3 && c.weight_bytes + c.patch_bytes + 8 * c.steps <= kWindowLds;
  const int64_t gemm_tiles = ((int64_t)g.batch * g.out_h * g.out_w + 127) / 128;
  const int64_t gemm_rounds = gemm_tiles < 128 ? 1 : (gemm_tiles + 511) / 512, slots = two ? 512 : 256, rounds = (c.tiles + slots - 1) / slots;
  return (float)rounds * (two ? 0.98f : window_blocks(g) == 3 ? 0.75f : 0.9f) < (float)gemm_rounds;
}
// Geometries that the kernel has a form for, images aside.
static inline bool window_form(const ConvGeom &g) {
  const int taps = g.kernel_h * g.kernel_w;
  if (g.in_c == 3 || g.in_c == 4)
    return g.out_c <= 128 && g.kernel_w <= 8 && g.kernel_h <= 16 && g.dilation_w == 1 &&
           g.kernel_h * (g.kernel_w * g.in_c > 16 ? 2 : 1) > 8;
  return (g.in_c & 15) == 0 && g.out_c <= 128 && taps > 1 && (int64_t)taps * g.in_c <= 2048;
}
// Whether images exist that choose_window has rectangles for: with half of a workgroup's pixels (choose_window), at least 8 wide
// (cut_window).  No rectangle of a 3x3 on 128 channels against 97 to 128, for one, fits beside the 144 KiB of its weights.
static inline bool window_fits(const ConvGeom &g) {
  if (!window_form(g)) return false;
  ConvGeom least = g;
  least.batch = 1;
  for (least.out_w = 8; least.out_w <= 64; ++least.out_w) {
    least.out_h = (32 * kWaves / 2 + least.out_w - 1) / least.out_w;
    WindowCut c;
    if (cut_window(least, &c) && c.tiles == 1) return true;
  }
  return false;
}
static inline bool choose_window(const ConvGeom &g, bool aligned, WindowCut *c) {
  const int64_t image = (int64_t)g.in_h * g.in_w * g.in_c;
  if (!window_form(g) || g.batch * image < 16 || image >= (int64_t)1 << 31) return false;
  if (!aligned && !packed_window(g)) return false;
  return cut_window(g, c) && c->tiles >= least_tiles(g) && wide_rounds_pay(g, *c) && c->tiles < 1 << 23 &&  // (2^32 threads)
         c->tiles * (32 * kWaves / 2) <= (int64_t)g.batch * g.out_h * g.out_w;
}

}  // namespace mi
