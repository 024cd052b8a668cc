// What the convolutions whose pixels are the matrix cores' row operand do with their products: a lane holds one output channel of
// 16 pixels per block of 32 channels, requantises them with that channel's parameters in registers, and a 4 x 4 byte
// transposition across neighbouring lanes makes dwords of four channels for the stores.
#pragma once

#include <type_traits>

#include "common.h"
#include "quant_math.h"

namespace mi {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t quad_transpose(uint32_t d, uint32_t sel1, uint32_t sel2) {
  const uint32_t p = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)d, 0xB1, 0xF, 0xF, true);  // lane ^ 1
  const uint32_t r = __builtin_amdgcn_perm(p, d, sel1);
  const uint32_t q = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r, 0x4E, 0xF, 0xF, true);  // lane ^ 2
  return __builtin_amdgcn_perm(q, r, sel2);
}

// Stores that stream are non-temporal: written out while the launch runs and not by the write-back of the L2s at its end.  For
// outputs that the L2s (32 MB) would still hold then: of larger ones most is out by that time, and a streamed one is not in the
// last-level cache for the launch that reads it.  And where a workgroup has all channels of its pixels, two whole blocks of them
// or more, so that its stores write whole lines.  us, temporal -> streamed: 32 x 224 x 224 x 3 -> 64, 7x7, stride 2 (26 MB) 17.4 -> 16.5,
// eight of them 6.35 -> 5.8; 16 x 112 x 112, 32 -> 96 8.0 -> 6.2, -> 160 12.5 -> 10.8; but -> 192 in groups of 96 14.5 -> 24.4.  Chains of
// stem, 1x1, depthwise and 1x1: on 112 x 112, 32 -> 128 -> 32 channels, 8 images 35.0 -> 31.5; 32 -> 192 -> 32, 32 images, all streamed
// 83 -> 94, those on 32 channels only 83 -> 91.
constexpr int64_t kStreamedMost = (int64_t)32 << 20;
inline bool conv_streams(int64_t pixels, int out_c, int blocks) {
  return blocks >= 2 && out_c == 32 * blocks && pixels * out_c <= kStreamedMost;
}

typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// One store of x at any address, non-temporal or not.  (The alignment belongs to the type that is stored through: as an argument's
// type it would be lost.)
template <bool STREAMED, typename T>
__device__ __forceinline__ void store_any(int8_t *to, T x) {
  typedef T any __attribute__((aligned(1)));
  if (STREAMED) {
    __builtin_nontemporal_store(x, reinterpret_cast<any *>(to));
  } else {
    *reinterpret_cast<any *>(to) = x;
  }
}

// What of a lane's 4 * OCB channels exists: all of them, whole quads, anything.
enum StoreForm { kWhole, kQuads, kBytes };

// How the convolutions requantise, see requant_form.
enum RequantForm { kGeneralForm, kCarryForm, kReluForm };

// kCarryForm: the one-multiply rounding without weight zero points, shifts up to 23 (so that the output range, shifted, is an int32).
// kReluForm: the same where no output is below the zero point (an activation): a negative x of RequantParams::fast2 ends below the
// range with [x >= 0] = 1 as it does with 0, so that pre + 1 goes into c2's high dword, and the carry and its add are not needed.
inline RequantForm requant_form(const RequantParams &rq) {
  if (rq.fast2 == 0 || rq.has_zw != 0 || rq.most_shift > 23) return kGeneralForm;
  return rq.amin >= rq.zo ? kReluForm : kCarryForm;
}

// The channel of a group of 32 * OCB that column r of channel block ob computes: either a lane's quads of channels (after the
// transposition), one per block, are neighbours in memory, or the blocks are, each with stores of its own.
__host__ __device__ __forceinline__ int column_channel(int ocb, int ob, int r, bool neighbours = true) {
  return neighbours ? 4 * ocb * (r >> 2) + 4 * ob + (r & 3) : 32 * ob + r;
}

// acc[ob][4 * q + e] is pixel 8 * q + 4 * h + e of 32, channel n0 + column_channel(OCB, ob, r, NEIGHBOURS); after the transposition a lane holds
// the quad of channels from n0 + column_channel(OCB, ob, r & ~3, NEIGHBOURS) of pixel 8 * q + 4 * h + (lane & 3).
// Vector instructions per quad: 23 with a shift and a clamp of its own for each output and a carry, 19 in kCarryForm and 15 in
// kReluForm, whose clamps come before the shift that saturates and packs.
template <int OCB, RequantForm FORM, bool NEIGHBOURS = true>
struct ChannelRequant {
  int32_t mult[OCB], bias[OCB], shift[OCB], lsh[OCB], zw[OCB];  // of this lane's channel of each block
  int32_t least[OCB], most[OCB];  // the output range before the shift
  uint64_t c2[OCB];
  uint32_t sel1, sel2;

  __device__ __forceinline__ ChannelRequant(const RequantParams &rq, int n0, int lane) {
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) {
      const int n = n0 + column_channel(OCB, ob, lane & 31, NEIGHBOURS);  // (the arrays are padded to a multiple of 256 channels)
      shift[ob] = rq.rshift[n];
      if (FORM == kGeneralForm) {
        const RequantChannel ch = rq.each[n];
        mult[ob] = ch.mult;
        bias[ob] = (int32_t)((uint32_t)ch.bias2 - kAccBias);
        lsh[ob] = ch.lshift();
        zw[ob] = ch.zw;
      } else {
        mult[ob] = (int32_t)rq.mult2[n];
        bias[ob] = rq.pre[n];
        const uint32_t hi = rq.c2hi[n] + (FORM == kReluForm ? (uint32_t)bias[ob] + 1 : 0);
        c2[ob] = (uint64_t)hi << 32 | rq.c2lo[n];
        least[ob] = (int32_t)((uint32_t)rq.amin << shift[ob]);
        most[ob] = (int32_t)((uint32_t)(rq.amax + 1) << shift[ob]) - 1;
      }
    }
    sel1 = (lane & 1) ? 0x03070105u : 0x06020400u, sel2 = (lane & 2) ? 0x03020706u : 0x05040100u;
  }
  __device__ __forceinline__ uint32_t four_channels(const RequantParams &rq, const v16i (&acc)[OCB], const v16i &sums, int q,
                                                    int ob) const {
    if (FORM == kGeneralForm) {
      int y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t v = (uint32_t)acc[ob][4 * q + e] - (uint32_t)sums[4 * q + e] * (uint32_t)zw[ob] + (uint32_t)bias[ob];
        int32_t t = rdiv_pot(srdhm((int32_t)(v << lsh[ob]), mult[ob]), shift[ob]);
        t = (int32_t)((uint32_t)t + (uint32_t)rq.zo);
        t = t < rq.amax ? t : rq.amax;
        y[e] = t > rq.amin ? t : rq.amin;
      }
      const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)y[1], (uint32_t)y[0], 0x0c0c0400u);
      const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)y[3], (uint32_t)y[2], 0x0c0c0400u);
      return quad_transpose(__builtin_amdgcn_perm(p23, p01, 0x05040100u), sel1, sel2);
    }
    int32_t t[4];
    if (FORM == kReluForm) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        t[e] = (int32_t)(((uint64_t)(uint32_t)acc[ob][4 * q + e] * (uint32_t)mult[ob] + c2[ob]) >> 32);
    } else {
      // one 64-bit multiply-add per output; its carry is the rounding's "+1 unless negative"
      uint64_t p2[4], carry[4], unused;
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
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) asm("v_med3_i32 %0, %0, %1, %2" : "+v"(t[e]) : "v"(least[ob]), "v"(most[ob]));
    const uint32_t p01 = (uint16_t)__builtin_amdgcn_ashr_pk_i8_i32((uint32_t)t[0], (uint32_t)t[1], (uint32_t)shift[ob]);
    const uint32_t p23 = (uint16_t)__builtin_amdgcn_ashr_pk_i8_i32((uint32_t)t[2], (uint32_t)t[3], (uint32_t)shift[ob]);
    return quad_transpose(__builtin_amdgcn_perm(p23, p01, 0x05040100u), sel1, sel2);
  }
  // quad q of each block, which is 4 * OCB neighbouring channels, to `to`; `have` of them exist
  template <StoreForm KIND, bool STREAMED>
  __device__ __forceinline__ void store(const RequantParams &rq, const v16i (&acc)[OCB], const v16i &sums, int q, int8_t *to,
                                        int have) const {
    uint32_t four[OCB];
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) four[ob] = four_channels(rq, acc, sums, q, ob);
    if constexpr (!NEIGHBOURS) {  // (whole blocks only)
#pragma unroll
      for (int ob = 0; ob < OCB; ++ob)
        if (KIND == kWhole || have > 0) store_any<STREAMED>(to + 32 * ob, four[ob]);
      return;
    }
    auto quad = [&](int ob) {
      if (KIND == kWhole || have >= 4 * ob + 4) {
        store_any<STREAMED>(to + 4 * ob, four[ob]);
      } else if (KIND == kBytes) {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (4 * ob + e < have) to[4 * ob + e] = (int8_t)(four[ob] >> (8 * e));
      }
    };
#pragma unroll
    for (int ob = 0; ob < OCB;) {
      if (ob + 4 <= OCB && KIND == kWhole) {
        store_any<STREAMED>(to + 4 * ob, v4u{four[ob], four[ob + 1], four[ob + 2], four[ob + 3]});
        ob += 4;
      } else if (ob + 2 <= OCB) {
        if (KIND == kWhole || have >= 4 * ob + 8) {
          store_any<STREAMED>(to + 4 * ob, v2u{four[ob], four[ob + 1]});
        } else {
          quad(ob);
          quad(ob + 1);
        }
        ob += 2;
      } else {
        quad(ob++);
      }
    }
  }
  // Calls store(kind, streamed) with constants, lanes without channels stay out of it where all pixels of the tile exist.  Bytes one
  // by one whenever a lane lacks channels took, 1x1 on 16 x 112 x 112 pixels, 24 -> 72 channels 9.8 us, this 7.7; 16 -> 48 7.2 / 6.0;
  // 16 -> 80 9.8 / 8.6.
  template <typename F>
  static __device__ __forceinline__ void in_form(bool all_pixels, int n0, int my_n, int out_c, bool streams, F store) {
    using std::integral_constant;
    if (out_c & 3) {
      store(integral_constant<StoreForm, kBytes>(), std::false_type());
    } else if (!all_pixels || (n0 + 32 * OCB > out_c && out_c % (4 * OCB) != 0)) {
      store(integral_constant<StoreForm, kQuads>(), std::false_type());
    } else if (streams) {
      store(integral_constant<StoreForm, kWhole>(), std::true_type());
    } else if (my_n < out_c) {
      store(integral_constant<StoreForm, kWhole>(), std::false_type());
    }
  }
};

// The compiler keeps the distance that a matrix product's result needs before the next instruction reads it, but not where that
// instruction is inline assembly, as above: 19 wait states after a 16-pass product.
template <int OCB>
__device__ __forceinline__ void wait_for_products(v16i (&acc)[OCB]) {
  asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]));
#pragma unroll
  for (int ob = 1; ob < OCB; ++ob) asm volatile("" : "+v"(acc[ob]));
}

}  // namespace mi
