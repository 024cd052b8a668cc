// What a kernel is launched with.
//
// The runtime writes a launch's arguments into device memory, and on many hosts that has a step in it: up to 112 bytes a launch
// costs the host 2.85 us, from 128 bytes on 3.55 (empty kernels, 16 to 768 bytes; where the bus is near 2.5 throughout).  A kernel
// that reads gridDim takes 72 bytes of hidden arguments more: with it the step is behind 40 bytes.  Launches of a few
// microseconds run at the host's pace, so their kernels get at most kShortArgs bytes, know their grid from their own sizes, and
// make the wider structures that the bodies work on from what they are given, in scalar registers.  (All but the groups of GEMMs and of
// more than two decode MatMuls, conv_window_kernel, the depthwise kernels other than conv_dw_rows_kernel, conv_smallk_kernel and im2col.)
// (Calls through Python, 240 to 256 bytes and hidden ones -> 64 to 112: FullConnection 128 x 768 x 768 4.55 -> 4.2 us, of which its
// kernel takes 3.9; the four convolutions of an image block 18.5 -> 16.5, their kernels 13.6.)
#pragma once

#include "common.h"

namespace mi {

constexpr size_t kShortArgs = 112;

// RequantParams of a matrix of n channels.
struct RequantCall {
  const RequantChannel *channels;
  int32_t zo, amin, amax;
  uint32_t forms;
  enum : uint32_t { kHasZw = 1, kFast = 2, kFast2 = 4 };
  static RequantCall of(const RequantParams &rq) {
    return RequantCall{rq.each, rq.zo, rq.amin, rq.amax, forms_of(rq)};
  }
  static uint32_t forms_of(const RequantParams &rq) {
    return (rq.has_zw != 0 ? kHasZw : 0u) | (rq.fast != 0 ? kFast : 0u) | (rq.fast2 != 0 ? kFast2 : 0u);
  }
  // Kernels that are short ask for all their arguments at once, with an empty asm of which they are the inputs: left to itself the compiler
  // loads some where they are used, one way to memory behind the other.
  __device__ __forceinline__ void load_now() const { asm volatile("" ::"s"(channels), "s"(zo), "s"(amin), "s"(amax), "s"(forms)); }
  __device__ __forceinline__ RequantParams open(int n) const {
    RequantParams rq{};
    rq.set_channels(channels, padded_channels(n));
    rq.zo = zo;
    rq.amin = amin;
    rq.amax = amax;
    rq.has_zw = (forms & kHasZw) != 0;
    rq.fast = (forms & kFast) != 0;
    rq.fast2 = (forms & kFast2) != 0;
    return rq;
  }
};

// DequantParams of a matrix of n channels whose rows of k bytes hold k - gap values.
struct DequantCall {
  const DequantChannel *channels;
  const mi_dq_params *qp_dev;
  float sx;
  int32_t zx, zw0;
  uint32_t forms;
  enum : uint32_t { kGap = 15, kHasBias = 16, kPerRow = 32, kActShift = 6 };
  static DequantCall of(const DequantParams &dq, int k) {
    return DequantCall{dq.each, dq.qp_dev, dq.sx, dq.zx, dq.zw0, forms_of(dq, k)};
  }
  static uint32_t forms_of(const DequantParams &dq, int k) {  // k: `deep` rounded up to at most a multiple of 16
    return (uint32_t)(k - dq.deep) | (dq.has_bias != 0 ? kHasBias : 0u) | (dq.per_row != 0 ? kPerRow : 0u) |
           (uint32_t)dq.act << kActShift;
  }
  __device__ __forceinline__ DequantParams open(int n, int k) const {
    DequantParams dq{};
    dq.set_channels(channels, padded_channels(n));
    dq.has_bias = (forms & kHasBias) != 0;
    dq.qp_dev = qp_dev;
    dq.sx = sx;
    dq.zx = zx;
    dq.zw0 = zw0;
    dq.deep = k - (int32_t)(forms & kGap);
    dq.act = (int32_t)(forms >> kActShift);
    dq.per_row = (forms & kPerRow) != 0;
    return dq;
  }
};

}  // namespace mi
