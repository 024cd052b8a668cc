// 1x1 convolutions against few output channels: the weights stay in LDS, the image goes straight from
// memory into the matrix cores' operand registers.
#include <string.h>

#include <type_traits>

#include "conv_store.h"
#include "launch_args.h"

namespace mi {

typedef v4i v4i_any __attribute__((aligned(1)));

// A workgroup holds the weights of OCB x 32 channels in LDS, in the order the MFMA operand takes them (1 KiB per 32 bytes
// of K and 32 channels), and its four waves walk tiles of 32 pixels each by itself, without barriers: a lane's 16 bytes of
// every 32-byte step of K are one load from the pixel's row, at whatever address that has, CH steps at a time, the next CH
// steps' loads in flight while this one's products run.  The GEMM's tiles stage both operands through LDS in barriered
// steps, fetch nothing for the next tile before they have stored this one, and are 128 or 256 channels wide however few
// there are; rows of any but a multiple of 16 bytes also had to be padded in a pass of their own.
// The pixels are the MFMA's row operand, see conv_store.h.
// Bound by the vector ALU (the requantisation, 4 instructions per output byte) and the stores where there are more channels than
// bytes of K, by memory where there are fewer.  us per launch, GEMM -> with a clamp, shift and carry of its own for each output
// and temporal stores of four bytes -> now: 16 x 112 x 112, 192 -> 32 channels 45.2 -> 10.7 -> 10.7, 32 -> 64 - -> 7.0 -> 5.5, 32 -> 128
// - -> 11.2 -> 8.4, 32 -> 192 21.0 -> 15.6 -> 13.5, 24 -> 72 - -> 8.9 -> 7.7; 8 x 115 x 115, 240 -> 40 26.5 -> 9.4 -> 9.2;
// 4 x 80 x 80, 72 -> 24 9.0 (in two launches) -> 3.5; one image of 112 x 112, where any launch takes most of it, 192 -> 32 3.7 -> 3.8.
// G: groups of OCB x 32 channels that a workgroup computes one after the other, see launch_conv_thin.
struct ConvThin {
  const int8_t *in;
  int64_t in_bytes;
  int k;       // contraction bytes
  int chunks;  // of CH steps; weights are zero from k on
  int out_c, pixels;
  bool streams;
  int step;         // tiles that all workgroups of a channel group do at once
  const int8_t *w;  // [32 channels][step][lane][16]
};
static_assert(sizeof(ConvThin) + sizeof(RequantCall) + sizeof(int8_t *) <= kShortArgs, "see launch_args.h");

template <int CH, int OCB, RequantForm FORM, bool NEIGHBOURS = true, int G = 1>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void conv_thin_kernel(ConvThin g, RequantCall call,
                                                                                              int8_t *__restrict__ out) {
  call.load_now();
  asm volatile("" ::"s"(g.in), "s"(g.in_bytes), "s"(g.k), "s"(g.chunks), "s"(g.out_c), "s"(g.pixels), "s"(g.step), "s"(g.w), "s"(out));
  const RequantParams rq = call.open(g.out_c);
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.y * (32 * OCB * G);
  const int tiles = (g.pixels + 31) >> 5, step = g.step;
  int tile = blockIdx.x * 4 + (tid >> 6);
  const int steps = g.chunks * CH;

  auto requant_of = [&](int grp) { return ChannelRequant<OCB, FORM, NEIGHBOURS>(rq, n0 + 32 * OCB * grp, lane); };
  const ChannelRequant<OCB, FORM, NEIGHBOURS> requant[2] = {requant_of(0), requant_of(G - 1)};

  int64_t at = 0;  // this lane's first byte of a tile
  auto locate = [&](int tl) {
    const int want = tl * 32 + r, p = want < g.pixels ? want : g.pixels - 1;
    at = (int64_t)p * g.k + 16 * h;
  };
  // Every load is a whole 16 bytes inside the tensor: one that would reach past its end is moved in (bytes past K meet zero
  // weights).
  const int64_t last = g.in_bytes - 16;
  auto fetch = [&](v4i (&x)[CH], int c) {
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int64_t off = at + (c * CH + s) * 32;
      x[s] = *reinterpret_cast<const v4i_any *>(g.in + (off < last ? off : last));
    }
  };

  {
    // From [32 channels][step][lane], front to back, into operand order [ob][step][lane], where the channels of a group are columns
    // of its blocks (ChannelRequant).  Fetched in operand order instead, 3 x 206 x 206, 376 -> 152 channels took 32.0 us, this 29.9;
    // 34 x 26 x 26, 336 -> 192 9.5 / 8.8.
    const int left = (g.out_c - n0 + 31) / 32, have = (left < OCB * G ? left : OCB * G) * steps;
    const v4i *src = reinterpret_cast<const v4i *>(g.w) + (int64_t)(n0 / 32) * steps * 64;
    v4i *dst = reinterpret_cast<v4i *>(lds);
#pragma unroll 4
    for (int i = __builtin_amdgcn_readfirstlane(tid >> 6); i < have; i += 4) {
      const int b = i / steps, s = i - b * steps, grp = b / OCB, n = 32 * (b - grp * OCB) + r;
      const int ob = NEIGHBOURS ? (n >> 2) % OCB : b, column = NEIGHBOURS ? 4 * (n / (4 * OCB)) + (n & 3) : r;
      dst[((grp * OCB + ob) * steps + s) * 64 + column + 32 * h] = src[i * 64 + lane];
    }
    __syncthreads();
  }
  if (tile >= tiles) return;
  v16i start;
#pragma unroll
  for (int e = 0; e < 16; ++e) start[e] = (int)kAccBias;
  locate(tile);
  v4i x[CH];
  fetch(x, 0);
  for (; tile < tiles; tile += step) {
    v16i acc[OCB], sums;
#pragma unroll
    for (int e = 0; e < 16; ++e) sums[e] = 0;
    v4i y[CH];
    auto take = [&](int c) {  // chunk c into y, the one behind it on its way
#pragma unroll
      for (int s = 0; s < CH; ++s) y[s] = x[s];
      const int64_t over = at + ((c + 1) * CH - 1) * 32 - last;
      if (__any(over > 0)) {  // a load that was moved in: move its bytes back
#pragma unroll
        for (int s = 0; s < CH; ++s) {
          const int64_t by = over - (CH - 1 - s) * 32;
          if (by > 0) {
            const unsigned __int128 v = __builtin_bit_cast(unsigned __int128, y[s]);
            y[s] = __builtin_bit_cast(v4i, by >= 16 ? (unsigned __int128)0 : v >> (8 * (int)by));
          }
        }
      }
      if (c + 1 < g.chunks) {
        fetch(x, c + 1);
      } else if (tile + step < tiles) {  // (wave-uniform)
        locate(tile + step);
        fetch(x, 0);
      }
    };
    auto products = [&](int c, int grp, auto first_c) {  // the first ones start the accumulators, from one register block for all
      const char *wl = lds + (grp * OCB * steps + c * CH) * 1024 + lane * 16;
#pragma unroll
      for (int s = 0; s < CH; ++s)
#pragma unroll
        for (int ob = 0; ob < OCB; ++ob)
          acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(y[s], *reinterpret_cast<const v4i *>(wl + (ob * steps + s) * 1024),
                                                          decltype(first_c)::value && s == 0 ? start : acc[ob], 0, 0, 0);
      if (FORM == kGeneralForm && rq.has_zw) {  // the pixels' input sums, in the accumulators' layout: against ones up to K
#pragma unroll
        for (int s = 0; s < CH; ++s) {
          v4i one;
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const int n = min(max(g.k - (c * CH + s) * 32 - 16 * h - 4 * d, 0), 4);
            one[d] = (int)(0x01010101u & (uint32_t)(((uint64_t)1 << (8 * n)) - 1));
          }
          sums = __builtin_amdgcn_mfma_i32_32x32x32_i8(y[s], one, sums, 0, 0, 0);
        }
      }
    };
    auto chunk = [&](int c, auto first_c) {
      take(c);
      products(c, 0, first_c);
    };
    const int first = tile * 32, my_p = first + 4 * h + (lane & 3);
    auto finish = [&](int grp) {
      wait_for_products(acc);
      const int g0 = n0 + 32 * OCB * grp, my_n = g0 + column_channel(OCB, 0, r & ~3, NEIGHBOURS);
      int8_t *dst = out + (int64_t)my_p * g.out_c + my_n;
      requant[grp].in_form(first + 32 <= g.pixels, g0, my_n, g.out_c, g.streams, [&](auto kind, auto streamed) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          requant[grp].template store<decltype(kind)::value, decltype(streamed)::value>(rq, acc, sums, q, dst + 8 * q * g.out_c,
                                                                                        my_p + 8 * q < g.pixels ? g.out_c - my_n : 0);
      });
    };
    // (One block of channels: few instructions to save, and a launch of so few that fetching the longer code shows:
    //  4 x 80 x 80, 72 -> 24 3.3 us, with the split forms 3.6.  Three blocks: 16 x 112 x 112, 32 -> 192 16.2 us, with them 14.7.)
    if constexpr (G == 2) {  // (a contraction of one chunk)
      take(0);
      products(0, 0, std::true_type());
      finish(0);
      products(0, 1, std::true_type());
      finish(1);
    } else if constexpr (OCB > 1) {
      chunk(0, std::true_type());
      for (int c = 1; c < g.chunks; ++c) chunk(c, std::false_type());
      finish(0);
    } else {
      acc[0] = start;
      for (int c = 0; c < g.chunks; ++c) chunk(c, std::false_type());
      finish(0);
    }
  }
}

// How a contraction of k bytes is cut: the number of steps per batch of loads that pads least (of those the largest).
struct ThinCut {
  int ch, chunks;
  int steps() const { return ch * chunks; }
};
static ThinCut thin_cut(int k) {
  const int steps = (k + 31) / 32;
  ThinCut t{0, 0};
  for (int ch = 4; ch > 0; --ch) {
    const int chunks = (steps + ch - 1) / ch;
    if (t.ch == 0 || chunks * ch < t.steps()) t.ch = ch, t.chunks = chunks;
  }
  return t;
}
// Blocks of 32 channels per workgroup: two or three, whichever pads less, so that a pixel's bytes serve 64 or 96 channels;
// one as long as a CU then gets no more than four workgroups, all of them at once: what such a launch lasts is one wave's chain of
// requantisations.  us at three blocks / one: 1 x 112 x 112, 32 -> 192 channels (588 workgroups of one block) 4.8 / 4.2;
// 4 x 80 x 80, 24 -> 72 (600) 4.6 / 3.8; at two / one: 1 x 64 x 64, 16 -> 64 (64) 3.8 / 3.1, and 8 x 115 x 115, 240 -> 40 (1654)
// 9.4 / 11.2.
static int thin_blocks(int64_t wgs, int oc) {
  const int blocks = (oc + 31) / 32;
  if (blocks == 1 || wgs * blocks <= 1024) return 1;
  return (blocks + 2) / 3 * 3 <= (blocks + 1) / 2 * 2 ? 3 : 2;
}

// Weights that leave a CU's LDS room for two workgroups or more, and few enough channels that re-reading the image for every
// 64 or 96 of them stays in the caches.
bool conv_thin_supported(int k, int oc) {
  return k <= 1024 && oc <= 256 && thin_cut(k).steps() * 1024 * thin_blocks((int64_t)1 << 30, oc) <= 64 * 1024;
}

// Weights [oc][k] -> ConvThin::w.
std::vector<int8_t> conv_thin_weights(const int8_t *w, int oc, int k) {
  const int steps = thin_cut(k).steps();
  std::vector<int8_t> out((size_t)((oc + 31) / 32) * steps * 1024, 0);
  for (int n = 0; n < oc; ++n)
    for (int k0 = 0; k0 < k; k0 += 16) {
      const int lane = n % 32 + 32 * (k0 / 16 % 2);
      memcpy(&out[(((size_t)(n / 32) * steps + k0 / 32) * 64 + lane) * 16], w + (size_t)n * k + k0,
             (size_t)(k - k0 < 16 ? k - k0 : 16));
    }
  return out;
}

// Groups of 64 channels, of pixels of 256 bytes, store faster block by block, 32 bytes a pixel, than with quads of both blocks as
// neighbours, which whole pixels of 64 gain by.  us, neighbours / blocks: 8 x 56 x 56, 64 -> 256 5.4 / 5.05; 16 x 80 x 80, 32 -> 256
// 12.8 / 11.4; 4 x 112 x 112 8.1 / 7.25; 32 x 28 x 28, 128 -> 256 6.45 / 6.35; but 32 x 56 x 56, 64 -> 128 7.95 / 8.05; 16 x 112 x 112,
// 32 -> 64 5.65 / 6.5.
template <int CH, int OCB>
static int launch_thin_pairs(const ConvThin &c, const RequantParams &rq, int8_t *out, dim3 grid, size_t lds, hipStream_t stream) {
  if (requant_form(rq) == kReluForm) {
    launch_kernel((conv_thin_kernel<CH, OCB, kReluForm, true, 2>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
  } else {
    launch_kernel((conv_thin_kernel<CH, OCB, kCarryForm, true, 2>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int CH, int OCB>
static int launch_thin(const ConvThin &c, const RequantParams &rq, int8_t *out, dim3 grid, size_t lds, hipStream_t stream) {
  const RequantForm form = requant_form(rq);
  if constexpr (OCB == 2) {
    if (form != kGeneralForm && c.out_c == 256) {
      if (form == kReluForm) {
        launch_kernel((conv_thin_kernel<CH, OCB, kReluForm, false>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
      } else {
        launch_kernel((conv_thin_kernel<CH, OCB, kCarryForm, false>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
      }
      MI_HIP_CHECK(hipGetLastError());
      return MI_OK;
    }
  }
  if (form == kReluForm) {
    launch_kernel((conv_thin_kernel<CH, OCB, kReluForm>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
  } else if (form == kCarryForm) {
    launch_kernel((conv_thin_kernel<CH, OCB, kCarryForm>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
  } else if constexpr (OCB <= 3) {
    launch_kernel((conv_thin_kernel<CH, OCB, kGeneralForm>), grid, dim3(256), lds, stream, c, RequantCall::of(rq), out);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

int launch_conv_thin(const int8_t *in, int64_t pixels, int k, int oc, const int8_t *w, const RequantParams &rq, int8_t *out,
                     hipStream_t stream) {
  if (!conv_thin_supported(k, oc) || pixels < 1 || pixels > kConvThinMostPixels || pixels * k < 16) {
    set_error("conv_thin: unsupported geometry k=%d oc=%d pixels=%lld", k, oc, (long long)pixels);
    return MI_PARAM_INVALID;
  }
  const ThinCut t = thin_cut(k);
  const int64_t wgs = (pixels + 127) / 128;
  const RequantForm form = requant_form(rq);
  const int blocks = (oc + 31) / 32;
  // Four or five whole blocks in one workgroup, whose stores then stream.  us, two groups -> this: 16 x 112 x 112, 32 -> 128 11.2 -> 8.9,
  // -> 160 15.3 -> 10.9; 16 x 56 x 56, 128 -> 128 6.0 -> 5.6.  Six (too few waves) 14.7 -> 22, channels short of five 10.4 -> 14.
  const bool rows = form != kGeneralForm && oc == 32 * blocks && blocks > 3 && blocks <= 5 && wgs * blocks > 1024 && t.steps() * blocks <= 64;
  const int ocb = rows ? blocks : thin_blocks(wgs, oc);
  // Two groups one after the other by the same wave, from the same operand registers, where the output is more than the L2s hold: a group's
  // 64 or 96 bytes of a pixel are parts of lines, of which the other group's workgroups write the rest when the line may have left.  us per
  // launch into changing memory, a workgroup per group / per pair: 16 x 112 x 112, 32 -> 192 20.9 / 14.1, 32 images 39.2 / 25.2, 24 -> 144
  // 35.2 / 20.9; image blocks whose expanded image stays in the last-level cache: 32 x 125 x 125, 40 -> 120 (60 MB) 82.3 / 73.5, 24 x 112 x 112
  // (36 MB) 55.4 / 51.4, 32 x 112 x 112, 24 -> 144 (58 MB) 72.3 / 69.2, 32 -> 192 (77 MB) 79.5 / 78.1, 16 images (38.5 MB) 47.0 / 47.2; outputs
  // that the L2s hold, with fewer waves at once 8 x 112 x 112, 32 -> 192 9.05 / 9.9, the block 31.7 / 33.8.
  const bool pairs = form != kGeneralForm && (ocb == 2 || ocb == 3) && (blocks + ocb - 1) / ocb == 2 && t.chunks == 1 &&
                     pixels * oc > kStreamedMost;
  const int in_wg = pairs ? 2 * ocb : ocb, groups = (blocks + in_wg - 1) / in_wg;
  // four workgroups per CU, which the LDS allows up to 40 KiB of weights; more would only load the weights more often
  const int most = (1024 + groups - 1) / groups;
  const dim3 grid((unsigned)(wgs < most ? wgs : most), (unsigned)groups);
  const ConvThin c{in, pixels * k, k, t.chunks, oc, (int)pixels, conv_streams(pixels, oc, ocb), 4 * (int)grid.x, w};
  const size_t lds = (size_t)t.steps() * in_wg * 1024;
#define MI_THIN(CH)                                                              \
  if (pairs && ocb == 2) return launch_thin_pairs<CH, 2>(c, rq, out, grid, lds, stream); \
  if (pairs) return launch_thin_pairs<CH, 3>(c, rq, out, grid, lds, stream);     \
  return ocb == 1   ? launch_thin<CH, 1>(c, rq, out, grid, lds, stream)          \
         : ocb == 2 ? launch_thin<CH, 2>(c, rq, out, grid, lds, stream)          \
         : ocb == 3 ? launch_thin<CH, 3>(c, rq, out, grid, lds, stream)          \
         : ocb == 4 ? launch_thin<CH, 4>(c, rq, out, grid, lds, stream)          \
                    : launch_thin<CH, 5>(c, rq, out, grid, lds, stream)
  switch (t.ch) {
    case 1: MI_THIN(1);
    case 2: MI_THIN(2);
    case 3: MI_THIN(3);
    default: MI_THIN(4);
  }
#undef MI_THIN
}

}  // namespace mi
