// Convolutions with a window of several taps on 16-channel-aligned images: the window's pixels and the weights in LDS.
#include <string.h>

#include <type_traits>

#include "conv_store.h"
#include "window_cut.h"

namespace mi {

// A workgroup of eight waves computes a rectangle of up to 256 output pixels for 32 x OCB channels, 32 pixels a wave.  It fetches
// the rectangle of input pixels under all their windows once, and the channels' weights, meets, and then every tap of every
// window is a fragment read from LDS at a shifted address: two barriers, where the gathering GEMM (gemm_conv_kernel) fetches the
// image once per tap in barriered steps of 64 bytes of K and waits out the latency of nine of them at 3x3 on 64 channels.
// LDS: weights in operand order, 1 KiB per 32 channels and 32 bytes of K; the input pixels row by row, each an odd number of
// 16-byte chunks apart, so that the 32 pixels of a fragment read (neighbours, or every second one) spread over the banks.
// K runs over taps, then channels, in chunks of 16; a step is two chunks, one for each half of the wave, whose LDS offsets come
// from a table.  The pixels are the MFMA's row operand, see conv_store.h.
// A workgroup lasts 4 to 6 us (fetch, products, requantisation and stores one after the other), which two per CU overlap in part: bound by
// that chain.  No unit is full: at the first of the shapes below the vector ALU is busy 41 % of the time, LDS 29 %, the matrix
// pipe 27 %, and waves wait 45 % of theirs.  us per launch, gathering GEMM -> this: 32 x 56 x 56,
// 64 -> 64 channels 11.9 -> 7.8; 512 x 14 x 14 11.6 -> 7.9; 64 x 56 x 56, 32 -> 32, stride 2 5.6 -> 4.5.  With every load waited for
// at the first barrier 0.9 more at the first of these, and then as four waves of 64 pixels each 2 % more, four of 32 in
// rectangles of 128 16 %, eight of 64 in 512 7 %.
//
// PACKED: the first layer's three or four channels, four bytes a pixel in LDS.  A window row is one or two chunks of four pixels
// (zero weights behind its last tap and in a fourth byte that is no channel), read at any pixel.  conv_rows_kernel takes such
// rows straight from the image in unaligned 16-byte loads, about 95 cycles of the address unit each; here a pixel's bytes are
// loaded once, four pixels a lane.  32 x 224 x 224 x 3 -> 64, 7x7, stride 2: 20.5 us -> 14.5 to 16.5, of which launch and prologue 5.9,
// the pixels 2, products 3, stores about 5 (26 MB); 296 vector instructions a wave keep the vector ALU busy 58 % of the time, fragment
// reads LDS 37 %.
//
// More than 64 channels (three and four blocks): the weights of a 3x3 on 96 channels alone are 81 KiB, so that one workgroup of eight waves
// has the CU.  Where the GEMM's tiles of 128 channels were a quarter empty and fetched every pixel nine times that is still far quicker:
// 32 x 56 x 56, 96 -> 96 21.7 -> 14.3, 80 -> 80 19.6 -> 14.1, 64 -> 96 16.0 -> 9.8, 64 -> 128 16.1 -> 13.2; packed, 32 x 224 x 224 x 3 -> 96,
// 7x7, stride 2 (conv_rows_kernel) 35.9 -> 19.6.
struct ConvWindow {
  const int8_t *in;
  const int8_t *in_last4;  // the tensor's last four bytes
  int in_h, in_w, in_c, out_h, out_w, out_c;
  int kernel_h, kernel_w, stride_h, stride_w, dil_h, dil_w, pad_u, pad_l;
  int tile_h, tile_w, tiles_x, tiles_y;  // output pixels of a workgroup
  int patch_h, patch_w;                  // input pixels under them
  int cc, pitch;                         // chunks per pixel, and from one pixel to the next in LDS
  int steps;                             // of 32 bytes of K
  int weight_bytes, patch_bytes;         // in LDS, multiples of 1 KiB
  bool streams;
  // ceil(2^32 / d): exact quotients for dividends < 2^16 (d >= 2; 0: d = 1)
  uint32_t magic_pitch, magic_patch_w, magic_tile_w, magic_cc, magic_kernel_w, magic_quads;
  uint32_t magic_tiles_x, magic_tiles_y;  // see magic31
  int shift_tiles_x, shift_tiles_y;
  const int8_t *w;       // [32 channels][step][lane][16]
  const int8_t *fill16;  // 16 bytes of what lies outside the image
};

__device__ __forceinline__ int quotient16(int p, uint32_t magic) { return magic == 0 ? p : (int)__umulhi((uint32_t)p, magic); }

typedef uint32_t u32_any __attribute__((aligned(1)));
typedef v4i v4i_4 __attribute__((aligned(4)));
typedef v4u v4u_any __attribute__((aligned(1)));

template <int OCB, bool PACKED, RequantForm FORM>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(OCB == 4 || (OCB == 3 && !PACKED) ? kWaves / 4 : kWaves / 2))) void conv_window_kernel(
    ConvWindow g, RequantParams rq, int8_t *__restrict__ out) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row_id = quotient31(blockIdx.x, g.magic_tiles_x, g.shift_tiles_x), b = quotient31(row_id, g.magic_tiles_y, g.shift_tiles_y);
  const int tx0 = (blockIdx.x - row_id * g.tiles_x) * g.tile_w, ty0 = (row_id - b * g.tiles_y) * g.tile_h;
  const ChannelRequant<OCB, FORM> requant(rq, 0, lane);

  auto to_lds = [](const void *from, void *wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                     (__attribute__((address_space(3))) void *)wave_base, 16, 0, 0);
  };
  char *patch = lds + g.weight_bytes;
  int *table = reinterpret_cast<int *>(patch + g.patch_bytes);
  // The first weights, the pixels, the last two loads of weights of each wave (three blocks: three): the products of the first weights
  // begin while those are on their way.
  constexpr int kLate = OCB == 3 ? 3 : 2, kLateSteps = kWaves * kLate / OCB;
  static_assert(PACKED || kLateSteps * OCB == kWaves * kLate, "every wave has as many late loads");
  const int early = PACKED ? 0 : max(g.steps - kLateSteps, 0);  // steps whose weights come first
  auto load_weights = [&](int from, int to) {
    for (int i = from * OCB + wave; i < to * OCB; i += kWaves) {
      to_lds(g.w + (i % OCB * g.steps + i / OCB) * 1024 + lane * 16, lds + i * 1024);
    }
  };
  // four pixels at a time; those of an image's edges, and the tensor's last ones, one by one
  auto load_patch = [&] {
    const int iy0 = ty0 * g.stride_h - g.pad_u, ix0 = tx0 * g.stride_w - g.pad_l, line = g.in_w * g.in_c;
    const int8_t *image = g.in + (int64_t)b * g.in_h * line;
    const int row_quads = g.patch_w >> 2, quads = g.patch_h * row_quads;
    for (int i = tid; i < quads; i += 64 * kWaves) {
      const int row = quotient16(i, g.magic_quads), iy = iy0 + row, ix = ix0 + 4 * (i - row * row_quads);
      const int8_t *want = image + iy * line + ix * g.in_c;
      v4u v;
      if ((unsigned)iy < (unsigned)g.in_h && ix >= 0 && ix + 4 <= g.in_w && want <= g.in_last4 - 12) {
        v = *reinterpret_cast<const v4u_any *>(want);
        if (g.in_c == 3)
          v = v4u{v[0], __builtin_amdgcn_alignbyte(v[1], v[0], 3), __builtin_amdgcn_alignbyte(v[2], v[1], 2), v[2] >> 8};
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bool inside = (unsigned)iy < (unsigned)g.in_h && (unsigned)(ix + u) < (unsigned)g.in_w;
          const int8_t *px = want + u * g.in_c, *from = px < g.in_last4 ? px : g.in_last4;
          v[u] = *reinterpret_cast<const u32_any *>(inside ? from : g.fill16) >> (inside ? (uint32_t)(px - from) * 8 : 0);
        }
      }
      reinterpret_cast<v4u *>(patch)[i] = v;
    }
  };
  load_weights(0, early);
  if constexpr (PACKED) {
    load_patch();
  } else {
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
  if constexpr (!PACKED) {
    // the table: where chunk f of a window lies from its first byte (behind the last chunk: that one again, against zeros)
    for (int f = tid; f < 2 * g.steps; f += 64 * kWaves) {
      const int ff = min(f, g.kernel_h * g.kernel_w * g.cc - 1), tap = quotient16(ff, g.magic_cc);
      const int kh = quotient16(tap, g.magic_kernel_w), kw = tap - kh * g.kernel_w;
      table[f] = ((kh * g.dil_h * g.patch_w + kw * g.dil_w) * g.pitch + ff - tap * g.cc) * 16;
    }
  }
  // Pixel t of the rectangle; where there is none, past the rectangle's last or outside the image, its first pixel again, which
  // is then computed and stored more than once.
  const int have_h = min(g.tile_h, g.out_h - ty0), have_w = min(g.tile_w, g.out_w - tx0);
  const int my_ty = quotient16(wave * 32 + r, g.magic_tile_w), my_tx = wave * 32 + r - my_ty * g.tile_w;
  const int my_px = my_ty < have_h && my_tx < have_w ? my_ty * g.stride_h * g.patch_w + my_tx * g.stride_w : 0;
  // Packed, a step is one window row of two chunks or two of one chunk (behind the last row: one more, against zeros).
  const int row_bytes = g.dil_h * g.patch_w * 4, step_bytes = g.cc == 2 ? row_bytes : 2 * row_bytes;
  const char *px = patch + (PACKED ? my_px * 4 + h * (g.cc == 2 ? 16 : row_bytes) : my_px * g.pitch * 16);
  v16i start;
#pragma unroll
  for (int e = 0; e < 16; ++e) start[e] = (int)kAccBias;
  // (in order: all but a wave's last kLate loads are in; with fewer steps than those load, all of them are waited for)
  if (early > 0) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLate) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }

  v16i acc[OCB];
  const char *wl = lds + lane * 16;
  auto read = [&](v4i &x, v4i (&w)[OCB], int s, int off) {
    if constexpr (PACKED) {
      x = *reinterpret_cast<const v4i_4 *>(px + off);
    } else {
      x = *reinterpret_cast<const v4i *>(px + off);
    }
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) w[ob] = *reinterpret_cast<const v4i *>(wl + (s * OCB + ob) * 1024);
  };
  auto mma = [&](const v4i &x, const v4i (&w)[OCB]) {
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, w[ob], acc[ob], 0, 0, 0);
  };
  auto offset = [&](int s) {
    if constexpr (PACKED) return s * step_bytes;
    return table[2 * s + h];
  };
  // steps [from, to), the first ones or not: operands one step ahead, offsets two
  auto run = [&](int from, int to, auto first_c) {
    v4i x0, w0[OCB], x1, w1[OCB];
    const int last = to - 1;
    read(x0, w0, from, offset(from));
    read(x1, w1, min(from + 1, last), offset(min(from + 1, last)));
    int off = offset(min(from + 2, last)), s = from + 1;
    if constexpr (decltype(first_c)::value) {  // the accumulators from one block of registers
#pragma unroll
      for (int ob = 0; ob < OCB; ++ob) acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0, w0[ob], start, 0, 0, 0);
    } else {
      mma(x0, w0);
    }
    for (; s < last; s += 2) {
      read(x0, w0, s + 1, off);
      off = offset(min(s + 2, last));
      mma(x1, w1);
      read(x1, w1, min(s + 2, last), off);
      off = offset(min(s + 3, last));
      mma(x0, w0);
    }
    if (s == last) mma(x1, w1);
  };
  if (early > 0) {
    run(0, early, std::true_type());
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    run(early, g.steps, std::false_type());
  } else {
    run(0, g.steps, std::true_type());
  }

  // acc[ob][4 * q + e]: pixel 32 * wave + 8 * q + 4 * h + e of the rectangle
  const int my_n = column_channel(OCB, 0, r & ~3), first = wave * 32 + 4 * h + (lane & 3);
  int8_t *rectangle = out + ((int64_t)(b * g.out_h + ty0) * g.out_w + tx0) * g.out_c;
  int ty = quotient16(first, g.magic_tile_w), tx = first - ty * g.tile_w;
  uint32_t at = (uint32_t)(ty * g.out_w + tx) * g.out_c;
  wait_for_products(acc);
  requant.in_form(true, 0, my_n, g.out_c, g.streams, [&](auto kind, auto streamed) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t to = (ty < have_h && tx < have_w ? at : 0u) + my_n;
      requant.template store<decltype(kind)::value, decltype(streamed)::value>(rq, acc, start, q, rectangle + to, g.out_c - my_n);
      tx += 8, at += 8 * g.out_c;  // (a rectangle is at least that wide)
      if (tx >= g.tile_w) tx -= g.tile_w, ++ty, at += (g.out_w - g.tile_w) * g.out_c;
    }
  });
}

// ---- host side -----------------------------------------------------------------------------------------------------
static uint32_t magic16(int d) { return d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + d - 1) / (uint64_t)d); }

static std::vector<int8_t> operand_order(const int8_t *w, int oc, int k) {
  const int steps = (k + 31) / 32, ocb = (oc + 31) / 32;
  std::vector<int8_t> out((size_t)ocb * steps * 1024, 0);
  for (int column = 0; column < 32 * ocb; ++column) {
    const int n = column_channel(ocb, column / 32, column % 32);
    if (n >= oc) continue;
    for (int k0 = 0; k0 < k; k0 += 16)
      memcpy(&out[(((size_t)(column / 32) * steps + k0 / 32) * 64 + column % 32 + 32 * (k0 / 16 % 2)) * 16],
             w + (size_t)n * k + k0, 16);
  }
  return out;
}

bool conv_window_weights_wanted(const ConvGeom &g) { return window_fits(g); }

std::vector<int8_t> conv_window_weights(const ConvGeom &g, const int8_t *w) {
  if (!packed_window(g)) return operand_order(w, g.out_c, g.kernel_h * g.kernel_w * g.in_c);
  const int k = g.kernel_h * row_chunks(g) * 16;
  std::vector<int8_t> wide((size_t)g.out_c * k, 0);
  for (int n = 0; n < g.out_c; ++n)
    for (int kh = 0; kh < g.kernel_h; ++kh)
      for (int kw = 0; kw < g.kernel_w; ++kw)
        memcpy(&wide[(size_t)n * k + kh * row_chunks(g) * 16 + kw * 4],
               w + (((size_t)n * g.kernel_h + kh) * g.kernel_w + kw) * g.in_c, g.in_c);
  return operand_order(wide.data(), g.out_c, k);
}

typedef void (*WindowKernel)(ConvWindow, RequantParams, int8_t *);
// [blocks of 32 channels - 1][packed][kReluForm]
static const WindowKernel kWindowKernels[4][2][2] = {
    {{conv_window_kernel<1, false, kCarryForm>, conv_window_kernel<1, false, kReluForm>},
     {conv_window_kernel<1, true, kCarryForm>, conv_window_kernel<1, true, kReluForm>}},
    {{conv_window_kernel<2, false, kCarryForm>, conv_window_kernel<2, false, kReluForm>},
     {conv_window_kernel<2, true, kCarryForm>, conv_window_kernel<2, true, kReluForm>}},
    {{conv_window_kernel<3, false, kCarryForm>, conv_window_kernel<3, false, kReluForm>},
     {conv_window_kernel<3, true, kCarryForm>, conv_window_kernel<3, true, kReluForm>}},
    {{conv_window_kernel<4, false, kCarryForm>, conv_window_kernel<4, false, kReluForm>},
     {conv_window_kernel<4, true, kCarryForm>, conv_window_kernel<4, true, kReluForm>}}};

// Dynamic LDS beyond 64 KiB has to be announced: cut_window gives all of them up to kWindowLds (packed, 8x8 windows at stride 8
// take 77 KiB) or kWindowLdsWide.
int conv_window_prepare_device() {
  for (const auto &of_blocks : kWindowKernels)
    for (const auto &of_packed : of_blocks)
      for (const WindowKernel kernel : of_packed)
        MI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         kWindowLdsWide));
  return MI_OK;
}

int launch_conv_window(const int8_t *in, const ConvGeom &g, const int8_t *fill16, const int8_t *w, const RequantParams &rq,
                       int8_t *out, hipStream_t stream, bool *taken) {
  WindowCut t;
  *taken = requant_form(rq) != kGeneralForm && choose_window(g, (reinterpret_cast<uintptr_t>(in) & 15) == 0, &t);
  if (!*taken) return MI_OK;
  const bool packed = packed_window(g);
  const int cc = packed ? row_chunks(g) : g.in_c / 16;
  ConvWindow c{};
  c.in = in;
  c.in_last4 = in + (int64_t)g.batch * g.in_h * g.in_w * g.in_c - 4;
  c.in_h = g.in_h, c.in_w = g.in_w, c.in_c = g.in_c, c.out_h = g.out_h, c.out_w = g.out_w, c.out_c = g.out_c;
  c.kernel_h = g.kernel_h, c.kernel_w = g.kernel_w, c.stride_h = g.stride_h, c.stride_w = g.stride_w;
  c.dil_h = g.dilation_h, c.dil_w = g.dilation_w, c.pad_u = g.pad_u, c.pad_l = g.pad_l;
  c.tile_h = t.tile_h, c.tile_w = t.tile_w, c.tiles_x = t.tiles_x, c.tiles_y = t.tiles_y;
  c.patch_h = t.patch_h, c.patch_w = t.patch_w, c.cc = cc, c.pitch = t.pitch, c.steps = t.steps;
  c.weight_bytes = t.weight_bytes, c.patch_bytes = t.patch_bytes;
  c.streams = conv_streams((int64_t)g.batch * g.out_h * g.out_w, g.out_c, window_blocks(g));
  c.magic_pitch = magic16(t.pitch), c.magic_patch_w = magic16(t.patch_w), c.magic_tile_w = magic16(t.tile_w);
  c.magic_cc = magic16(cc), c.magic_kernel_w = magic16(g.kernel_w), c.magic_quads = magic16(t.patch_w / 4);
  c.w = w, c.fill16 = fill16;
  magic31(t.tiles_x, &c.magic_tiles_x, &c.shift_tiles_x);
  magic31(t.tiles_y, &c.magic_tiles_y, &c.shift_tiles_y);
  const size_t lds = (size_t)t.weight_bytes + t.patch_bytes + 8 * (size_t)t.steps;
  const dim3 grid((unsigned)t.tiles), threads(64 * kWaves);
  const WindowKernel kernel = kWindowKernels[window_blocks(g) - 1][packed][requant_form(rq) == kReluForm];
  launch_kernel(kernel, grid, threads, lds, stream, c, rq, out);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
