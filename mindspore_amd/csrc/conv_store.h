// What the convolutions whose pixels are the matrix cores' row operand do with their products: a lane holds one output channel of
// 16 pixels per block of 32 channels, requantises them with that channel's parameters in registers, and a 4 x 4 byte
// transposition across neighbouring lanes makes dwords of four channels for the stores.
#pragma once

#include "common.h"
#include "quant_math.h"

namespace mi {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Quotients of p < 2^31 by d >= 1 as umulhi(2 p, magic) >> shift, with 2^(shift - 1) < d <= 2^shift and
// magic = ceil(2^(31 + shift) / d): the product is p / d + p * e / (d * 2^(31 + shift)), e = magic * d - 2^(31 + shift) < 2^shift,
// and the second term stays below 1 / d.
inline void magic31(int d, uint32_t *magic, int *shift) {
  int s = 0;
  while (((int64_t)1 << s) < d) ++s;
  *shift = s;
  *magic = (uint32_t)((((uint64_t)1 << (31 + s)) + (uint32_t)d - 1) / (uint32_t)d);
}

__device__ __forceinline__ int quotient31(int p, uint32_t magic, int shift) { return (int)(__umulhi(2 * (uint32_t)p, magic) >> shift); }

__device__ __forceinline__ uint32_t quad_transpose(uint32_t d, uint32_t sel1, uint32_t sel2) {
  const uint32_t p = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)d, 0xB1, 0xF, 0xF, true);  // lane ^ 1
  const uint32_t r = __builtin_amdgcn_perm(p, d, sel1);
  const uint32_t q = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x4E, 0xF, 0xF, true);  // lane ^ 2
  return __builtin_amdgcn_perm(q, r, sel2);
}

// acc[ob][4 * q + e] is pixel 8 * q + 4 * h + e of 32, channel n0 + 32 * ob + r; after the transposition a lane holds channels
// r & ~3 .. + 3 of pixel 8 * q + 4 * h + (lane & 3).
// FAST: the one-multiply rounding form without weight zero points (RequantParams::fast2, !has_zw).
template <int OCB, bool FAST>
struct ChannelRequant {
  int32_t mult[OCB], bias[OCB], shift[OCB], lsh[OCB], zw[OCB];  // of this lane's channel of each block
  uint64_t c2[OCB];
  int amin_v, amax_v;
  uint32_t sel1, sel2;

  __device__ __forceinline__ ChannelRequant(const RequantParams &rq, int n0, int lane) {
    const int r = lane & 31;
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) {
      const int n = n0 + ob * 32 + r;  // (the arrays are padded to a multiple of 256 channels)
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
    amin_v = rq.amin, amax_v = rq.amax;
    asm volatile("" : "+v"(amin_v), "+v"(amax_v));  // kept in vector registers, as v_med3 wants them
    sel1 = (lane & 1) ? 0x03070105u : 0x06020400u, sel2 = (lane & 2) ? 0x03020706u : 0x05040100u;
  }
  __device__ __forceinline__ uint32_t four_channels(const RequantParams &rq, const v16i (&acc)[OCB], const v16i &sums, int q,
                                                    int ob) const {
    int y[4];
    if (FAST) {
      // one 64-bit multiply-add per output; its carry is the rounding's "+1 unless negative"
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
    return quad_transpose(__builtin_amdgcn_perm(p23, p01, 0x05040100u), sel1, sel2);
  }
};

// The compiler keeps the distance that a matrix product's result needs before the next instruction reads it, but not where that
// instruction is inline assembly, as above: 19 wait states after a 16-pass product.
template <int OCB>
__device__ __forceinline__ void wait_for_products(v16i (&acc)[OCB]) {
  if constexpr (OCB == 1) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]));
  if constexpr (OCB == 2) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]), "+v"(acc[1]));
}

// four channels of a pixel, as far as they exist
__device__ __forceinline__ void store_channels(int8_t *to, uint32_t four, int have) {
  typedef uint32_t u32_any __attribute__((aligned(1)));
  if (have >= 4) {
    *reinterpret_cast<u32_any *>(to) = four;
  } else {
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (e < have) to[e] = (int8_t)(four >> (8 * e));
  }
}

}  // namespace mi
