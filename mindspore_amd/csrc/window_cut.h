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

// Up to 128 channels, which one workgroup computes (more would fetch the pixels again), rectangles for two CUs in three (65 to 96 channels, and
// some first layers: three in eight), and at least half of their pixels there.  Time of this relative to the gathering GEMM, 3x3: workgroups 112 1.01, 128 1.02, 140 1.02,
// 160 1.02, 168 0.88 0.91, 192 0.87, 196 0.89, 224 0.87, 256 0.77, 448 0.75, 1024 0.70; stride 2 256 0.74; 5x5 128 0.84, 256 0.73.
// Rectangles filled to 0.77 0.77, 0.56 0.87, 0.39 0.90 to 1.05, 0.25 1.43, 0.19 1.40 to 2.1.
// 65 to 96 channels, of which the GEMM's 128-channel tiles leave a quarter and more empty, already from 96 workgroups: 96 -> 96 56 1.02,
// 98 0.84, 112 0.86, 224 0.72, 448 0.66, 64 -> 96 56 1.10, 112 0.90, 448 0.61, 32 -> 72 896 0.55; 97 to 128: 64 -> 128 112 1.03, 128 1.04,
// 224 0.84, 448 0.82, 32 -> 128 252 0.89.
// Three or four channels: windows for which conv_rows_kernel makes five or more loads.  Time relative to that one, us: 7x7 on 3
// channels -> 64, 49 workgroups 4.42 / 4.42, 98 4.46 / 4.48, 196 6.2 / 4.65, 392 8.55 / 6.05, 784 12.2 / 9.55, 1568 20.5 / 16.5;
// -> 96, 49 4.82 / 4.89, 98 6.71 / 5.06, 1568 35.9 / 19.6, -> 128, 98 6.78 / 5.73, 1568 38.1 / 24.0;
// 5x5 on 4 (five loads) 4.85 / 4.4 and 14.8 / 14.7, -> 96, 90 workgroups 5.10 / 4.55; 5x5 on 3 (three) 4.15 / 4.18; 3x3 on 3 (two)
// 5.17 / 5.55 and 7.7 / 8.8.  97 to 127 channels, whose stores have ragged ends in every fourth block: 96 to 167 workgroups 0.61 to 1.23 of the
// time, on average 1.03, from 168 on 0.49 to 1.1 and 0.85; 112 and 128 channels 0.83 and 0.68.
constexpr int kWindowLeastTiles = 168, kWindowLeastWideTiles = 96;
static inline int least_tiles(const ConvGeom &g) {
  return window_blocks(g) == 3 || (window_blocks(g) == 4 && packed_window(g) && g.out_c % 16 == 0) ? kWindowLeastWideTiles : kWindowLeastTiles;
}
// More than 64 channels against windows of 16-channel-aligned images: what both take, in us, least squares over 1599 shapes (windows of 2 to 25
// taps, strides 1 to 3, 14 x 14 to 112 x 112 images, 32 to 1300 rectangles; median error 3 to 5 %).  Mostly one workgroup has a CU, and what counts
// is how many rounds of them there are beside those of the GEMM's 128 x 128 tiles, two a CU.  A rectangle holds every pixel under it, also those
// that strides leave out, which beside few taps is more than the GEMM fetches; and channels that are no multiple of 16 have ragged stores.
// Of the 1599, by rounds alone 994 ran here, at 0.85 of the GEMM's time on average and 117 of them at 1.03 to 1.53; by this 829, at 0.81, twelve at
// 1.04 to 1.14; 17 that took 0.86 to 0.95 are given up.  us, GEMM / this: 32 x 56 x 56, 96 -> 96 21.7 / 14.3; not taken: 1x2, stride 2,
// 67 x 40 x 40, 128 -> 96 5.96 / 7.73; 1x3, stride 2, 23 x 112 x 112, 64 -> 80 9.77 / 12.28; 3x3 12 x 80 x 80, 32 -> 97 14.4 / 16.1.
static inline bool window_is_quicker(const ConvGeom &g, const WindowCut &c) {
  struct Cost {
    float launch, whole, part, patch, k, ragged, bytes;
  };
  constexpr Cost kTwo{2.5f, 1.06f, 2.8f, 0.033f, 0.66f, 0.69f, 1.38f}, kThree{1.9f, 2.55f, 0.1f, 0.026f, 0.51f, 0.25f, 0.92f},
      kFour{2.2f, 2.7f, -0.3f, 0.027f, 0.68f, 1.88f, 1.79f};
  if (window_blocks(g) < 3 || packed_window(g)) return true;
  // (four blocks take the registers of one workgroup)
  const bool two = window_blocks(g) == 3 && c.weight_bytes + c.patch_bytes + 8 * c.steps <= kWindowLds;
  const Cost &cost = two ? kTwo : window_blocks(g) == 3 ? kThree : kFour;
  const auto whole = [](int64_t tiles, int slots) { return (float)((tiles + slots - 1) / slots); };
  const int slots = two ? 512 : 256;
  const int64_t gemm_tiles = ((int64_t)g.batch * g.out_h * g.out_w + 127) / 128;
  const float k = (float)(g.kernel_h * g.kernel_w * g.in_c) / 100.0f, ragged = g.out_c % 16 != 0, bytes = g.out_c % 4 != 0;
  const float rounds = (float)c.tiles / (float)slots, mixed = 0.6f * whole(c.tiles, slots) + 0.4f * rounds;
  const float here = cost.launch + cost.whole * whole(c.tiles, slots) + rounds * (cost.part + cost.ragged * ragged + cost.bytes * bytes) +
                     mixed * (cost.patch * (float)(c.patch_bytes / 1024) + cost.k * k);
  if (gemm_tiles < 128) {  // (64 x 64 there)
    const float part = (float)gemm_tiles / 128.0f;
    return here < 3.88f + 0.18f * part + k * (0.35f + 0.105f * part);
  }
  const float gemm_rounds = (float)gemm_tiles / 512.0f, gemm_whole = whole(gemm_tiles, 512);
  const float passed_over = (float)(g.stride_h * g.stride_w * g.in_c) / 100.0f;  // (lines of the image of which the taps read a part)
  return here < 2.61f + 1.41f * gemm_whole + gemm_rounds * (2.11f + 1.35f * ragged + 0.48f * bytes + 0.24f * passed_over) +
                    k * (0.274f * gemm_whole + 0.546f * gemm_rounds + 0.186f * std::min(2.0f * gemm_rounds, 1.0f));
}
// Geometries that the kernel has a form for, images aside.
static inline bool window_form(const ConvGeom &g) {
  const int taps = g.kernel_h * g.kernel_w;
  if (g.in_c == 3 || g.in_c == 4)
    return g.out_c <= 128 && g.kernel_w <= 8 && g.kernel_h <= 16 && g.dilation_w == 1 &&
           g.kernel_h * (g.kernel_w * g.in_c > 16 ? 2 : 1) > 8;
  return (g.in_c & 15) == 0 && g.out_c <= 128 && taps > 1 && (int64_t)taps * g.in_c <= 2048;
}
// Images in rectangles that are quicker than what else there is.
static inline bool rectangles_pay(const ConvGeom &g, WindowCut *c) {
  return cut_window(g, c) && c->tiles >= least_tiles(g) && window_is_quicker(g, *c) && c->tiles < 1 << 23 &&  // (2^32 threads)
         c->tiles * (32 * kWaves / 2) <= (int64_t)g.batch * g.out_h * g.out_w;
}
// Whether there are such images, asked of as many as make one round of rectangles to eight, each a rectangle of at least half of a workgroup's
// pixels.  No rectangle of a 3x3 on 128 channels against 97 to 128, for one, fits beside the 144 KiB of its weights.
static inline bool window_fits(const ConvGeom &g) {
  if (!window_form(g)) return false;
  ConvGeom one = g;
  for (one.out_w = 8; one.out_w <= 64; ++one.out_w)
    for (one.out_h = 32 * kWaves / one.out_w; 2 * one.out_h * one.out_w >= 32 * kWaves; --one.out_h) {
      WindowCut c;
      one.batch = 1;
      if (!cut_window(one, &c) || c.tiles != 1) continue;
      for (const int tiles : {kWindowLeastTiles, 256, 512, 768, 2048}) {
        c.tiles = one.batch = tiles;
        if (window_is_quicker(one, c)) return true;
      }
    }
  return false;
}
static inline bool choose_window(const ConvGeom &g, bool aligned, WindowCut *c) {
  const int64_t image = (int64_t)g.in_h * g.in_w * g.in_c;
  if (!window_form(g) || g.batch * image < 16 || image >= (int64_t)1 << 31) return false;
  return (aligned || packed_window(g)) && rectangles_pay(g, c);
}

}  // namespace mi
