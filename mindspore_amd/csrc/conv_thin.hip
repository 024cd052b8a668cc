// 1x1 convolutions against few output channels: the weights stay in LDS, the image goes straight from
// memory into the matrix cores' operand registers.
#include <string.h>

#include <type_traits>

#include "common.h"
#include "quant_math.h"

namespace mi {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef v4i v4i_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));

// A workgroup holds the weights of OCB x 32 channels in LDS, in the order the MFMA operand takes them (1 KiB per 32 bytes
// of K and 32 channels), and its four waves walk tiles of 32 pixels each by itself, without barriers: a lane's 16 bytes of
// every 32-byte step of K are one load from the pixel's row, at whatever address that has, CH steps at a time, the next CH
// steps' loads in flight while this one's products run.  The GEMM's tiles stage both operands through LDS in barriered
// steps, fetch nothing for the next tile before they have stored this one, and are 128 or 256 channels wide however few
// there are; rows of any but a multiple of 16 bytes also had to be padded in a pass of their own.
// The pixels are the MFMA's row operand: a lane ends up with one output channel of 16 pixels per block of 32 channels, with
// its requantisation parameters in registers, and a 4 x 4 byte transposition across neighbouring lanes makes dwords of four
// channels for the stores (as in conv_rows_kernel).
// Bound by the vector ALU (the requantisation, 7 instructions per output byte) where there are more channels than bytes of
// K, by memory where there are fewer.  us per launch, before -> now: 16 x 112 x 112, 192 -> 32 channels 45.2 -> 10.6,
// 32 -> 192 21.0 -> 14.7; 8 x 115 x 115, 240 -> 40 26.5 -> 9.6; 4 x 80 x 80, 72 -> 24 9.0 (in two launches) -> 3.5; one
// image of 112 x 112, where any launch takes most of it, 192 -> 32 3.7 -> 3.8.
// Windows of several taps stay with the gathering GEMM: 32 x 56 x 56 x 64, 3x3, took 13.6 us in this form against 14.0, one
// such image 6.2 against 5.1, stride 2 10.6 against 7.1.
struct ConvThin {
  const int8_t *in;
  int64_t in_bytes;
  int k;       // contraction bytes
  int chunks;  // of CH steps; weights are zero from k on
  int out_c, pixels;
  const int8_t *w;  // [32 channels][step][lane][16]
};

__device__ __forceinline__ uint32_t thin_quad_transpose(uint32_t d, uint32_t sel1, uint32_t sel2) {
  const uint32_t p = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)d, 0xB1, 0xF, 0xF, false);  // lane ^ 1
  const uint32_t r = __builtin_amdgcn_perm(p, d, sel1);
  const uint32_t q = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x4E, 0xF, 0xF, false);  // lane ^ 2
  return __builtin_amdgcn_perm(q, r, sel2);
}

// FAST: the one-multiply rounding form without weight zero points (RequantParams::fast2, !has_zw).
template <int CH, int OCB, bool FAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void conv_thin_kernel(ConvThin g, RequantParams rq,
                                                                                              int8_t *__restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.y * (32 * OCB);
  const int tiles = (g.pixels + 31) >> 5, step = gridDim.x * 4;
  int tile = blockIdx.x * 4 + (tid >> 6);
  const int steps = g.chunks * CH;

  // this lane's channel of each block (the arrays are padded to a multiple of 256 channels)
  int32_t mult[OCB], bias[OCB], shift[OCB], lsh[OCB], zw[OCB];
  uint64_t c2[OCB];
#pragma unroll
  for (int ob = 0; ob < OCB; ++ob) {
    const int n = n0 + ob * 32 + r;
    shift[ob] = rq.rshift[n];
    if (FAST) {
      mult[ob] = (int32_t)rq.mult2[n];
      c2[ob] = (uint64_t)rq.c2hi[n] << 32 | rq.c2lo[n];
      bias[ob] = rq.pre[n];
    } else {
      mult[ob] = rq.mult[n];
      bias[ob] = (int32_t)((uint32_t)rq.bias2[n] - kAccBias);
      lsh[ob] = rq.lshift[n];
      zw[ob] = rq.zw[n];
    }
  }
  int amin_v = rq.amin, amax_v = rq.amax;
  asm volatile("" : "+v"(amin_v), "+v"(amax_v));  // kept in vector registers, as v_med3 wants them
  const uint32_t sel1 = (lane & 1) ? 0x03070105u : 0x06020400u, sel2 = (lane & 2) ? 0x03020706u : 0x05040100u;

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
    const v4i *src = reinterpret_cast<const v4i *>(g.w + (int64_t)(n0 / 32) * steps * 1024);
    const int have = min(OCB, (g.out_c - n0 + 31) / 32) * steps * 64;  // (the last group of blocks may reach past the weights)
    v4i *dst = reinterpret_cast<v4i *>(lds);
#pragma unroll 4
    for (int i = tid; i < have; i += 256) dst[i] = src[i];
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
    auto chunk = [&](int c, auto first_c) {  // the first one starts the accumulators, from one register block for all
      v4i y[CH];
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
      const char *wl = lds + c * CH * 1024 + lane * 16;
#pragma unroll
      for (int s = 0; s < CH; ++s)
#pragma unroll
        for (int ob = 0; ob < OCB; ++ob)
          acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(y[s], *reinterpret_cast<const v4i *>(wl + (ob * steps + s) * 1024),
                                                          decltype(first_c)::value && s == 0 ? start : acc[ob], 0, 0, 0);
      if (!FAST && rq.has_zw) {  // the pixels' input sums, in the accumulators' layout: against ones up to K
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
    // (One block of channels: few instructions to save, and a launch of so few that fetching the longer code shows:
    //  4 x 80 x 80, 72 -> 24 3.3 us, with the split forms 3.6.  Three blocks: 16 x 112 x 112, 32 -> 192 16.2 us, with them 14.7.)
    if constexpr (OCB > 1) {
      chunk(0, std::true_type());
      for (int c = 1; c < g.chunks; ++c) chunk(c, std::false_type());
    } else {
      acc[0] = start;
      for (int c = 0; c < g.chunks; ++c) chunk(c, std::false_type());
    }
    // (the wait states that a matrix product's result needs before inline assembly reads it, as in conv_rows_kernel)
    if constexpr (OCB == 1) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]));
    if constexpr (OCB == 2) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]), "+v"(acc[1]));
    if constexpr (OCB == 3) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]));
    // acc[ob][4 * q + e] is pixel 8 * q + 4 * h + e of the tile, channel n0 + 32 * ob + r; after the transposition this
    // lane holds channels r & ~3 .. + 3 of pixel 8 * q + 4 * h + (lane & 3)
    const int first = tile * 32;
    const bool whole = first + 32 <= g.pixels && n0 + 32 * OCB <= g.out_c;
    const int my_n = n0 + (r & ~3), my_p = first + 4 * h + (lane & 3);
    int8_t *dst = out + (int64_t)my_p * g.out_c + my_n;
    auto store = [&](auto whole_c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int ob = 0; ob < OCB; ++ob) {
        int y[4];
        if (FAST) {
          uint64_t p2[4], carry[4], unused;
          int32_t t[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            asm("v_mad_u64_u32 %0, %1, %2, %3, %4"
                : "=&v"(p2[e]), "=s"(carry[e])
                : "v"(acc[ob][4 * q + e]), "v"(mult[ob]), "v"(c2[ob]));
#pragma unroll
          for (int e = 0; e < 4; ++e)
            asm("v_addc_co_u32_e64 %0, %1, %2, %3, %4"
                : "=v"(t[e]), "=s"(unused)
                : "v"((int32_t)(p2[e] >> 32)), "v"(bias[ob]), "s"(carry[e]));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            t[e] >>= shift[ob];
            asm("v_med3_i32 %0, %1, %2, %3" : "=v"(y[e]) : "v"(t[e]), "v"(amin_v), "v"(amax_v));
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            uint32_t v = (uint32_t)acc[ob][4 * q + e] - (uint32_t)sums[4 * q + e] * (uint32_t)zw[ob] + (uint32_t)bias[ob];
            int32_t t = rdiv_pot(srdhm((int32_t)(v << lsh[ob]), mult[ob]), shift[ob]);
            t = (int32_t)((uint32_t)t + (uint32_t)rq.zo);
            t = t < rq.amax ? t : rq.amax;
            y[e] = t > rq.amin ? t : rq.amin;
          }
        }
        const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)y[1], (uint32_t)y[0], 0x0c0c0400u);
        const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)y[3], (uint32_t)y[2], 0x0c0c0400u);
        const uint32_t four = thin_quad_transpose(__builtin_amdgcn_perm(p23, p01, 0x05040100u), sel1, sel2);
        int8_t *to = dst + 8 * q * g.out_c + 32 * ob;
        if (decltype(whole_c)::value || (my_p + 8 * q < g.pixels && my_n + 32 * ob + 4 <= g.out_c)) {
          *reinterpret_cast<u32_any *>(to) = four;
        } else if (my_p + 8 * q < g.pixels) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (my_n + 32 * ob + e < g.out_c) to[e] = (int8_t)(four >> (8 * e));
        }
      }
    }
    };
    if (OCB > 1 && whole) {
      store(std::true_type());
    } else {
      store(std::false_type());
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

template <int CH, int OCB>
static int launch_thin(const ConvThin &c, const RequantParams &rq, int8_t *out, dim3 grid, size_t lds, hipStream_t stream) {
  if (rq.fast2 != 0 && rq.has_zw == 0) {
    hipLaunchKernelGGL((conv_thin_kernel<CH, OCB, true>), grid, dim3(256), lds, stream, c, rq, out);
  } else {
    hipLaunchKernelGGL((conv_thin_kernel<CH, OCB, false>), grid, dim3(256), lds, stream, c, rq, out);
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
  const ConvThin c{in, pixels * k, k, t.chunks, oc, (int)pixels, w};
  const int64_t wgs = (pixels + 127) / 128;
  const int ocb = thin_blocks(wgs, oc), groups = (oc + 32 * ocb - 1) / (32 * ocb);
  // four workgroups per CU, which the LDS allows up to 40 KiB of weights; more would only load the weights more often
  const int most = (1024 + groups - 1) / groups;
  const dim3 grid((unsigned)(wgs < most ? wgs : most), (unsigned)groups);
  const size_t lds = (size_t)t.steps() * ocb * 1024;
#define MI_THIN(CH)                                                              \
  return ocb == 1   ? launch_thin<CH, 1>(c, rq, out, grid, lds, stream)          \
         : ocb == 2 ? launch_thin<CH, 2>(c, rq, out, grid, lds, stream)          \
                    : launch_thin<CH, 3>(c, rq, out, grid, lds, stream)
  switch (t.ch) {
    case 1: MI_THIN(1);
    case 2: MI_THIN(2);
    case 3: MI_THIN(3);
    default: MI_THIN(4);
  }
#undef MI_THIN
}

}  // namespace mi
