// Convolutions with a window of several taps on 16-channel-aligned images: the window's pixels and the weights in LDS.
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "conv_store.h"

namespace mi {

// A workgroup of eight waves computes a rectangle of up to 256 output pixels for 32 x OCB channels, 32 pixels a wave.  It fetches
// the rectangle of input pixels under all their windows once, and the channels' weights, meets, and then every tap of every
// window is a fragment read from LDS at a shifted address: two barriers, where the gathering GEMM (gemm_conv_kernel) fetches the
// image once per tap in barriered steps of 64 bytes of K and waits out the latency of nine of them at 3x3 on 64 channels.
// LDS: weights in operand order, 1 KiB per 32 channels and 32 bytes of K; the input pixels row by row, each an odd number of
// 16-byte chunks apart, so that the 32 pixels of a fragment read (neighbours, or every second one) spread over the banks.
// K runs over taps, then channels, in chunks of 16; a step is two chunks, one for each half of the wave, whose LDS offsets come
// from a table.  The pixels are the MFMA's row operand and the stores those of conv_rows_kernel.
// A workgroup lasts about 4 us (fetch 1.5, products 1, requantisation and stores 1.5), which two per CU overlap: bound by that
// chain up to 512 workgroups and by LDS reads and the vector ALU beyond.  us per launch, gathering GEMM -> this: 32 x 56 x 56,
// 64 -> 64 channels 12.1 -> 9.2; 512 x 14 x 14 12.6 -> 9.7; 512 x 512, 16 -> 16 10.0 -> 7.4; 64 x 28 x 28, 32 -> 64, 5x5 9.3 -> 6.7;
// 64 x 56 x 56, 32 -> 32, stride 2 5.8 -> 5.0.  With every load waited for at the first barrier 9.8 at the first of these, and
// then as four waves of 64 pixels each 10.0, four of 32 in rectangles of 128 11.4, eight of 64 in 512 10.5.
struct ConvWindow {
  const int8_t *in;
  int in_h, in_w, in_c, out_h, out_w, out_c;
  int kernel_h, kernel_w, stride_h, stride_w, dil_h, dil_w, pad_u, pad_l;
  int tile_h, tile_w, tiles_x, tiles_y;  // output pixels of a workgroup
  int patch_h, patch_w;                  // input pixels under them
  int cc, pitch;                         // chunks per pixel, and from one pixel to the next in LDS
  int steps;                             // of 32 bytes of K
  int weight_bytes, patch_bytes;         // in LDS, multiples of 1 KiB
  uint32_t magic_pitch, magic_patch_w, magic_tile_w;  // ceil(2^32 / d): exact quotients for dividends < 2^16 (d >= 2; 0: d = 1)
  uint32_t magic_tiles_x, magic_tiles_y;  // see magic31
  int shift_tiles_x, shift_tiles_y;
  const int8_t *w;       // [32 channels][step][lane][16]
  const int8_t *fill16;  // 16 bytes of what lies outside the image
};

__device__ __forceinline__ int quotient16(int p, uint32_t magic) { return magic == 0 ? p : (int)__umulhi((uint32_t)p, magic); }

constexpr int kWaves = 8;

template <int OCB>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kWaves / 2))) void conv_window_kernel(ConvWindow g, RequantParams rq,
                                                                                                int8_t *__restrict__ out) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row_id = quotient31(blockIdx.x, g.magic_tiles_x, g.shift_tiles_x), b = quotient31(row_id, g.magic_tiles_y, g.shift_tiles_y);
  const int tx0 = (blockIdx.x - row_id * g.tiles_x) * g.tile_w, ty0 = (row_id - b * g.tiles_y) * g.tile_h;
  const ChannelRequant<OCB, true> requant(rq, 0, lane);

  auto to_lds = [](const void *from, void *wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                     (__attribute__((address_space(3))) void *)wave_base, 16, 0, 0);
  };
  char *patch = lds + g.weight_bytes;
  int *table = reinterpret_cast<int *>(patch + g.patch_bytes);
  // The first weights, the pixels, the last two loads of weights of each wave: the products of the first weights begin while
  // those are on their way.
  constexpr int kLate = 2, kLateSteps = kWaves * kLate / OCB;
  const int early = max(g.steps - kLateSteps, 0);  // steps whose weights come first
  auto load_weights = [&](int from, int to) {
    for (int i = from * OCB + wave; i < to * OCB; i += kWaves) {
      to_lds(g.w + (i % OCB * g.steps + i / OCB) * 1024 + lane * 16, lds + i * 1024);
    }
  };
  load_weights(0, early);
  {
    const int iy0 = ty0 * g.stride_h - g.pad_u, ix0 = tx0 * g.stride_w - g.pad_l;
    const int8_t *image = g.in + (int64_t)b * g.in_h * g.in_w * g.in_c;
    const int chunks = g.patch_h * g.patch_w * g.pitch;
    for (int i = wave * 64; i < chunks; i += 64 * kWaves) {
      const int at = i + lane, px = quotient16(at, g.magic_pitch), c = at - px * g.pitch;
      const int row = quotient16(px, g.magic_patch_w), iy = iy0 + row, ix = ix0 + px - row * g.patch_w;
      const bool inside = at < chunks && c < g.cc && (unsigned)iy < (unsigned)g.in_h && (unsigned)ix < (unsigned)g.in_w;
      to_lds(inside ? image + ((int64_t)iy * g.in_w + ix) * g.in_c + c * 16 : g.fill16, patch + i * 16);
    }
  }
  load_weights(early, g.steps);
  // the table: where chunk f of a window lies from its first byte (behind the last chunk: that one again, against zeros)
  const int taps = g.kernel_h * g.kernel_w;
  for (int f = tid; f < 2 * g.steps; f += 64 * kWaves) {
    const int ff = min(f, taps * g.cc - 1), tap = ff / g.cc, kh = tap / g.kernel_w, kw = tap - kh * g.kernel_w;
    table[f] = ((kh * g.dil_h * g.patch_w + kw * g.dil_w) * g.pitch + ff - tap * g.cc) * 16;
  }
  // Pixel t of the rectangle; where there is none, past the rectangle's last or outside the image, its first pixel again, which
  // is then computed and stored more than once.
  auto locate = [&](int t, int *ty, int *tx) {
    *ty = quotient16(t, g.magic_tile_w);
    *tx = t - *ty * g.tile_w;
    if (*ty >= g.tile_h || ty0 + *ty >= g.out_h || tx0 + *tx >= g.out_w) *ty = *tx = 0;
  };
  int my_ty, my_tx;
  locate(wave * 32 + r, &my_ty, &my_tx);
  const char *px = patch + (my_ty * g.stride_h * g.patch_w + my_tx * g.stride_w) * g.pitch * 16;
  v16i start;
#pragma unroll
  for (int e = 0; e < 16; ++e) start[e] = (int)kAccBias;
  // (in order: all but a wave's last two loads are in; with fewer steps than those load, all of them are waited for)
  if (early > 0) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLate) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }

  v16i acc[OCB];
  const char *wl = lds + lane * 16;
  auto read = [&](v4i &x, v4i (&w)[OCB], int s, int off) {
    x = *reinterpret_cast<const v4i *>(px + off);
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) w[ob] = *reinterpret_cast<const v4i *>(wl + (s * OCB + ob) * 1024);
  };
  auto mma = [&](const v4i &x, const v4i (&w)[OCB]) {
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, w[ob], acc[ob], 0, 0, 0);
  };
#pragma unroll
  for (int ob = 0; ob < OCB; ++ob) acc[ob] = start;
  // steps [from, to): operands one step ahead, offsets two
  auto run = [&](int from, int to) {
    v4i x0, w0[OCB], x1, w1[OCB];
    const int last = to - 1;
    read(x0, w0, from, table[2 * from + h]);
    int off = table[2 * min(from + 1, last) + h];
    int s = from;
    for (; s < last; s += 2) {
      read(x1, w1, s + 1, off);
      off = table[2 * min(s + 2, last) + h];
      mma(x0, w0);
      read(x0, w0, min(s + 2, last), off);
      off = table[2 * min(s + 3, last) + h];
      mma(x1, w1);
    }
    if (s == last) mma(x0, w0);
  };
  if (early > 0) {
    run(0, early);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
  run(early, g.steps);

  // acc[ob][4 * q + e]: pixel 32 * wave + 8 * q + 4 * h + e of the rectangle, channel 32 * ob + r
  const int my_n = r & ~3;
  int8_t *image_out = out + (int64_t)b * g.out_h * g.out_w * g.out_c;
  wait_for_products(acc);
  auto store = [&](auto whole_c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int ty, tx;
      locate(wave * 32 + 8 * q + 4 * h + (lane & 3), &ty, &tx);
      int8_t *to = image_out + ((int64_t)(ty0 + ty) * g.out_w + tx0 + tx) * g.out_c + my_n;
#pragma unroll
      for (int ob = 0; ob < OCB; ++ob) {
        const uint32_t four = requant.four_channels(rq, acc, start, q, ob);
        store_channels(to + 32 * ob, four, decltype(whole_c)::value ? 4 : g.out_c - my_n - 32 * ob);
      }
    }
  };
  if (32 * OCB <= g.out_c) {
    store(std::true_type());
  } else {
    store(std::false_type());
  }
}

// ---- host side -----------------------------------------------------------------------------------------------------
static uint32_t magic16(int d) { return d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + d - 1) / (uint64_t)d); }

std::vector<int8_t> conv_window_weights(const int8_t *w, int oc, int k) {
  const int steps = (k + 31) / 32;
  std::vector<int8_t> out((size_t)((oc + 31) / 32) * steps * 1024, 0);
  for (int n = 0; n < oc; ++n)
    for (int k0 = 0; k0 < k; k0 += 16)
      memcpy(&out[(((size_t)(n / 32) * steps + k0 / 32) * 64 + n % 32 + 32 * (k0 / 16 % 2)) * 16], w + (size_t)n * k + k0, 16);
  return out;
}

constexpr int kWindowLds = 80 << 10;  // two workgroups per CU
struct WindowCut {
  int tile_h, tile_w, tiles_x, tiles_y, patch_h, patch_w, pitch, steps, weight_bytes, patch_bytes;
  int64_t tiles;
};
// The rectangles of an image that need the fewest workgroups, and of those the fewest input pixels; false if none fits.
static bool cut_window(const ConvGeom &g, WindowCut *best) {
  const int cc = g.in_c / 16, most = 32 * kWaves;  // (tile_w <= most)
  WindowCut c{};
  c.pitch = cc | 1;
  c.steps = (g.kernel_h * g.kernel_w * cc + 1) / 2;
  c.weight_bytes = (g.out_c > 32 ? 2 : 1) * c.steps * 1024;
  best->tiles = 0;
  for (int nx = (g.out_w + 63) / 64, last = std::min(64, (g.out_w + 7) / 8); nx <= last; ++nx) {  // 8 to 64 pixels wide
    c.tile_w = (g.out_w + nx - 1) / nx;
    c.tiles_x = (g.out_w + c.tile_w - 1) / c.tile_w;
    c.tile_h = std::min(most / c.tile_w, g.out_h);
    c.tiles_y = (g.out_h + c.tile_h - 1) / c.tile_h;
    c.tile_h = (g.out_h + c.tiles_y - 1) / c.tiles_y;
    const int64_t ph = (int64_t)(c.tile_h - 1) * g.stride_h + (int64_t)(g.kernel_h - 1) * g.dilation_h + 1;
    const int64_t pw = (int64_t)(c.tile_w - 1) * g.stride_w + (int64_t)(g.kernel_w - 1) * g.dilation_w + 1;
    if (ph > 4096 || pw > 4096) continue;
    c.patch_h = (int)ph;
    c.patch_w = (int)pw;
    const int64_t bytes = (ph * pw * c.pitch * 16 + 1023) / 1024 * 1024;  // (hence fewer than 2^16 chunks)
    if (c.weight_bytes + bytes + 8 * c.steps > kWindowLds) continue;
    c.patch_bytes = (int)bytes;
    c.tiles = (int64_t)c.tiles_x * c.tiles_y * g.batch;
    if (best->tiles == 0 || c.tiles < best->tiles || (c.tiles == best->tiles && c.patch_bytes < best->patch_bytes)) *best = c;
  }
  return best->tiles != 0;
}

// Up to 64 channels, which one workgroup computes (more would fetch the pixels again), rectangles for two CUs in three, and at
// least half of their pixels there.  Time of this relative to the gathering GEMM, 3x3: workgroups 112 1.01, 128 1.02, 140 1.02,
// 160 1.02, 168 0.88 0.91, 192 0.87, 196 0.89, 224 0.87, 256 0.77, 448 0.75, 1024 0.70; stride 2 256 0.74; 5x5 128 0.84, 256 0.73.
// Rectangles filled to 0.77 0.77, 0.56 0.87, 0.39 0.90 to 1.05, 0.25 1.43, 0.19 1.40 to 2.1.  Before its waits were cut, against
// 65 to 128 channels 0.99 to 1.24.
constexpr int kWindowLeastTiles = 168;
bool conv_window_weights_wanted(const ConvGeom &g) {
  return (g.in_c & 15) == 0 && g.out_c <= 64 && g.kernel_h * g.kernel_w > 1 && (int64_t)g.kernel_h * g.kernel_w * g.in_c <= 2048;
}
static bool choose_window(const ConvGeom &g, const void *in, WindowCut *c) {
  return conv_window_weights_wanted(g) && (reinterpret_cast<uintptr_t>(in) & 15) == 0 && cut_window(g, c) && c->tiles >= kWindowLeastTiles &&
         c->tiles * (32 * kWaves / 2) <= (int64_t)g.batch * g.out_h * g.out_w && c->tiles < 1 << 23;  // (2^32 threads)
}

int conv_window_prepare_device() {  // (more than 64 KiB of dynamic LDS)
  for (const void *kernel : {reinterpret_cast<const void *>(conv_window_kernel<1>), reinterpret_cast<const void *>(conv_window_kernel<2>)})
    MI_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kWindowLds));
  return MI_OK;
}

int launch_conv_window(const int8_t *in, const ConvGeom &g, const int8_t *fill16, const int8_t *w, const RequantParams &rq,
                       int8_t *out, hipStream_t stream, bool *taken) {
  WindowCut t;
  *taken = choose_window(g, in, &t);
  if (!*taken) return MI_OK;
  ConvWindow c{in, g.in_h, g.in_w, g.in_c, g.out_h, g.out_w, g.out_c, g.kernel_h, g.kernel_w, g.stride_h, g.stride_w, g.dilation_h,
               g.dilation_w, g.pad_u, g.pad_l, t.tile_h, t.tile_w, t.tiles_x, t.tiles_y, t.patch_h, t.patch_w, g.in_c / 16, t.pitch,
               t.steps, t.weight_bytes, t.patch_bytes, magic16(t.pitch), magic16(t.patch_w), magic16(t.tile_w), 0, 0, 0, 0, w, fill16};
  magic31(t.tiles_x, &c.magic_tiles_x, &c.shift_tiles_x);
  magic31(t.tiles_y, &c.magic_tiles_y, &c.shift_tiles_y);
  const size_t lds = (size_t)t.weight_bytes + t.patch_bytes + 8 * (size_t)t.steps;
  const dim3 grid((unsigned)t.tiles), threads(64 * kWaves);
  if (g.out_c > 32) {
    hipLaunchKernelGGL((conv_window_kernel<2>), grid, threads, lds, stream, c, rq, out);
  } else {
    hipLaunchKernelGGL((conv_window_kernel<1>), grid, threads, lds, stream, c, rq, out);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
