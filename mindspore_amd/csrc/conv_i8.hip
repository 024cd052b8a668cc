// Data-movement kernels in front of the GEMM for Conv2D int8, and the depthwise convolution.
//   pad_rows : [rows][k] -> zero-padded [rows][k16]           (activations whose K is not a multiple of 16)
//   im2col   : NHWC image -> [pixels][k16], K order (kh, kw, ic) as Im2ColPackUnitInt8Opt lays rows out
//              (reference mindspore/ccsrc/plugin/device/cpu/kernel/nnacl/int8/conv_int8.c:758-807); taps outside
//              the image take `fill`: the input zero point for the im2col convolution (conv_int8.c:877) and 0 for
//              the strided/padded 1x1 convolution (Conv1x1InputPack into a zeroed buffer,
//              .../nnacl/base/conv1x1_base.c:19-40, mindspore/lite/src/litert/kernel/cpu/int8/
//              convolution_1x1_int8.cc:396)
//   conv_dw  : depthwise conv + requantisation (ConvDwInt8 / ConvDwInt8Post,
//              .../nnacl/int8/conv_depthwise_int8.c:24-140); conv_dw_rows: the same with stride 1 and int8 weights, four
//              taps per instruction
//   conv_rows : first-layer convolutions (few input channels) in one launch, window rows straight from the image
//   conv_smallk : what is left with kernel_h * kernel_w * in_c <= 64 in one launch, gathered byte by byte
// The first three are HBM/latency bound byte movers: one thread produces 16 contiguous output bytes (or one output
// element for the depthwise kernel, consecutive threads on consecutive channels) so stores coalesce.
#include <string.h>

#include "conv_store.h"
#include "launch_args.h"

namespace mi {

typedef int v2i __attribute__((ext_vector_type(2)));

typedef v4i v4i_any __attribute__((aligned(1)));

// One 16-byte chunk per thread, taken with one load at whatever byte address the row length puts it (16 byte loads took
// 3.4 us for 333 x 1000, now 2.4, which is what any launch takes).  The last, partial chunk of a row is the row's last 16
// bytes shifted down, so nothing past the tensor is read, nor anything before it.
__global__ __launch_bounds__(256) void pad_rows_kernel(const int8_t *__restrict__ src, int64_t src_ld, int64_t total,
                                                       int k, int8_t *__restrict__ dst, int chunks_per_row, int threads) {
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += threads) {
    const int64_t row = total < 0x7fffffff ? (int64_t)((uint32_t)idx / (uint32_t)chunks_per_row)
                                           : idx / chunks_per_row;
    const int at = (int)(idx - row * chunks_per_row) * 16, have = k - at;
    const int8_t *s = src + row * src_ld + at;
    v4i v = {0, 0, 0, 0};
    if (have >= 16) {
      v = *reinterpret_cast<const v4i_any *>(s);
    } else if (row * src_ld + k >= 16) {
      const unsigned __int128 x = __builtin_bit_cast(unsigned __int128, *reinterpret_cast<const v4i_any *>(s + have - 16));
      v = __builtin_bit_cast(v4i, x >> (8 * (16 - have)));
    } else {  // rows within the first 16 bytes of the tensor
#pragma unroll
      for (int j = 0; j < 15; ++j)
        if (j < have) v[j >> 2] |= (int)((uint32_t)(uint8_t)s[j] << (8 * (j & 3)));
    }
    *reinterpret_cast<v4i *>(dst + idx * 16) = v;
  }
}

int launch_pad_rows(const int8_t *src, int64_t src_ld, int rows, int k, int8_t *dst, int k16, hipStream_t stream) {
  const int64_t total = (int64_t)rows * (k16 >> 4), want = (total + 255) / 256;
  const int wgs = (int)(want < 1048576 ? want : 1048576);
  launch_kernel(pad_rows_kernel, dim3(wgs), dim3(256), 0, stream, src, src_ld, total, k, dst, k16 >> 4, 256 * wgs);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

__global__ __launch_bounds__(256) void im2col_kernel(const int8_t *__restrict__ in, ConvGeom g, int fill,
                                                     int8_t *__restrict__ dst, int k16) {
  const int kdim = g.kernel_h * g.kernel_w * g.in_c;
  const int chunks_per_row = k16 >> 4;
  const int64_t pixels = (int64_t)g.batch * g.out_h * g.out_w;
  const int64_t total = pixels * chunks_per_row;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = idx / chunks_per_row;
    const int ch = (int)(idx - p * chunks_per_row);
    const int b = (int)(p / ((int64_t)g.out_h * g.out_w));
    const int rem = (int)(p - (int64_t)b * g.out_h * g.out_w);
    const int oh = rem / g.out_w, ow = rem - oh * g.out_w;
    const int ih0 = oh * g.stride_h - g.pad_u, iw0 = ow * g.stride_w - g.pad_l;
    const int8_t *img = in + (int64_t)b * g.in_h * g.in_w * g.in_c;
    union {
      v4i v;
      int8_t b[16];
    } u;
    int kk = ch * 16;
    int tap = kk / g.in_c, ic = kk - tap * g.in_c;
    int kh = tap / g.kernel_w, kw = tap - kh * g.kernel_w;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      int8_t val = 0;
      if (kk + j < kdim) {
        const int ih = ih0 + kh * g.dilation_h, iw = iw0 + kw * g.dilation_w;
        const bool inside = ih >= 0 && ih < g.in_h && iw >= 0 && iw < g.in_w;
        val = inside ? img[((int64_t)ih * g.in_w + iw) * g.in_c + ic] : (int8_t)fill;
      }
      u.b[j] = val;
      if (++ic == g.in_c) {
        ic = 0;
        if (++kw == g.kernel_w) {
          kw = 0;
          ++kh;
        }
      }
    }
    *reinterpret_cast<v4i *>(dst + p * k16 + ch * 16) = u.v;
  }
}

int launch_im2col(const int8_t *in, const ConvGeom &g, int fill, int8_t *dst, int k16, hipStream_t stream) {
  const int64_t total = (int64_t)g.batch * g.out_h * g.out_w * (k16 >> 4);
  const int64_t want = (total + 255) / 256;
  const int blocks = (int)(want < 1 ? 1 : (want > 1048576 ? 1048576 : want));
  launch_kernel(im2col_kernel, dim3(blocks), dim3(256), 0, stream, in, g, fill, dst, k16);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

// Dense convolution with a short contraction (kernel_h * kernel_w * in_c <= 64) that neither conv_rows_kernel nor the
// gathering GEMM takes, without an im2col buffer and its extra launch.  One wave produces 32 output pixels x
// all output channels with v_mfma_i32_32x32x32_i8: lane (r, h) gathers bytes [16h, 16h + 16) of every 32-byte K step
// of pixel r straight from the image, in the K order (kh, kw, ic) of Im2ColPackUnitInt8Opt (conv_int8.c:758-807),
// taps outside the image read as `fill` (conv_int8.c:877), bytes past K as 0; the weights come from the packed
// row-major copy (zero filled past K).  Same exact epilogue as the GEMM.
template <int KSTEPS, int OCB>
__global__ __launch_bounds__(256) void conv_smallk_kernel(const int8_t *__restrict__ in, ConvGeom g, int fill,
                                                          int k_true, const int8_t *__restrict__ w, int ldw,
                                                          RequantParams rq, int8_t *__restrict__ out) {
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 32;
  const int64_t pixels = (int64_t)g.batch * g.out_h * g.out_w;
  if (first >= pixels) return;  // the whole wave
  const bool live = first + r < pixels;
  const int64_t p = live ? first + r : pixels - 1;
  const int b = (int)(p / ((int64_t)g.out_h * g.out_w));
  const int rem = (int)(p - (int64_t)b * g.out_h * g.out_w);
  const int oh = rem / g.out_w, ow = rem - oh * g.out_w;
  const int ih0 = oh * g.stride_h - g.pad_u, iw0 = ow * g.stride_w - g.pad_l;
  const int8_t *img = in + (int64_t)b * g.in_h * g.in_w * g.in_c;

  // The requantisation parameters of the lane's channels, a block of 32 output channels at a time: prm[q][..] are
  // channels 32 * ob + 8 * q + 4 * h .. + 3.  Fetched without a branch on the channel or on the kind of parameters
  // (the arrays are padded to a multiple of 256 channels and all exist) and all sixteen-plus-four at once: the first
  // block's before the gather, so that they arrive behind it.  Fetched where they are used, one group of four
  // channels after the other and behind the branches of the previous group's arithmetic, they were four round trips
  // in a row at the end of a 32-channel stem.
  const int n_pad = padded_channels(g.out_c);
  v4i prm[4][5];
  auto fetch_params = [&](int ob) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int nb = ob * 32 + q * 8 + h * 4;
      prm[q][0] = *reinterpret_cast<const v4i *>(rq.mult(n_pad) + nb);
      prm[q][1] = *reinterpret_cast<const v4i *>(rq.bias2(n_pad) + nb);
      prm[q][2] = *reinterpret_cast<const v4i *>(rq.rshift + nb);
      prm[q][3] = *reinterpret_cast<const v4i *>(rq.zw + nb);
      prm[q][4] = *reinterpret_cast<const v4i *>(rq.lshift(n_pad) + nb);
    }
  };
  fetch_params(0);

  union Frag {
    v4i v;
    int8_t b[16];
  };
  Frag x[KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) {
    const int k0 = 32 * s + 16 * h;
    int tap = k0 / g.in_c, ic = k0 - tap * g.in_c;
    int kh = tap / g.kernel_w, kw = tap - kh * g.kernel_w;
    // no load is predicated: a byte that is not wanted is fetched from the pixel's image origin and replaced, so
    // that all sixteen loads are in flight together
    int8_t raw[16];
    int other[16];  // -1: take the loaded byte; otherwise the value to use instead
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int ih = ih0 + kh * g.dilation_h, iw = iw0 + kw * g.dilation_w;
      const bool in_k = k0 + i < k_true;
      const bool inside = ih >= 0 && ih < g.in_h && iw >= 0 && iw < g.in_w;
      const int64_t off = (in_k && inside) ? ((int64_t)ih * g.in_w + iw) * g.in_c + ic : 0;
      raw[i] = img[off];
      other[i] = in_k ? (inside ? -1 : (fill & 0xff)) : 0;
      const bool wrap_c = ic + 1 == g.in_c;
      const bool wrap_w = wrap_c && kw + 1 == g.kernel_w;
      ic = wrap_c ? 0 : ic + 1;
      kw = wrap_w ? 0 : (wrap_c ? kw + 1 : kw);
      kh = wrap_w ? kh + 1 : kh;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) x[s].b[i] = other[i] < 0 ? raw[i] : (int8_t)other[i];
  }

  v16i acc[OCB];
#pragma unroll
  for (int ob = 0; ob < OCB; ++ob)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[ob][e] = 0;
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
    for (int ob = 0; ob < OCB; ++ob) {
      const v4i wf = *reinterpret_cast<const v4i *>(w + (int64_t)(ob * 32 + r) * ldw + 32 * s + 16 * h);
      acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf, x[s].v, acc[ob], 0, 0, 0);
    }
  int rowsum = 0;
  if (rq.has_zw) {
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      rowsum = __builtin_amdgcn_sdot4(x[s].v.x, 0x01010101, rowsum, false);
      rowsum = __builtin_amdgcn_sdot4(x[s].v.y, 0x01010101, rowsum, false);
      rowsum = __builtin_amdgcn_sdot4(x[s].v.z, 0x01010101, rowsum, false);
      rowsum = __builtin_amdgcn_sdot4(x[s].v.w, 0x01010101, rowsum, false);
    }
    rowsum += __shfl_xor(rowsum, 32);
  }

  // acc[ob][4 * q + e] is output channel 32 * ob + 8 * q + 4 * h + e of pixel r
#pragma unroll
  for (int ob = 0; ob < OCB; ++ob) {
    if (ob > 0) fetch_params(ob);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int nb = ob * 32 + q * 8 + h * 4;
      const v4i mult4 = prm[q][0], bias4 = prm[q][1], e4 = prm[q][2], zw4 = prm[q][3], ls4 = prm[q][4];
      union {
        uint32_t u;
        int8_t b[4];
      } o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t v = (uint32_t)acc[ob][q * 4 + e];
        if (rq.has_zw) v -= (uint32_t)rowsum * (uint32_t)zw4[e];
        v += (uint32_t)bias4[e];
        int32_t t;
        if (rq.fast) {
          t = rdiv_pot_fast(srdhm_nosat((int32_t)v, mult4[e]), e4[e], (1 << e4[e]) >> 1);
        } else {
          t = rdiv_pot(srdhm((int32_t)(v << ls4[e]), mult4[e]), e4[e]);
        }
        t = (int32_t)((uint32_t)t + (uint32_t)rq.zo);
        t = t < rq.amax ? t : rq.amax;
        t = t > rq.amin ? t : rq.amin;
        o.b[e] = (int8_t)t;
      }
      if (live && nb < g.out_c) *reinterpret_cast<uint32_t *>(out + p * g.out_c + nb) = o.u;
    }
  }
}

int launch_conv_smallk(const int8_t *in, const ConvGeom &g, int fill, int k_true, const int8_t *w, int ldw,
                       const RequantParams &rq, int8_t *out, hipStream_t stream) {
  const int64_t pixels = (int64_t)g.batch * g.out_h * g.out_w;
  if (k_true < 1 || k_true > 64 || g.out_c < 4 || g.out_c > 128 || (g.out_c & 3) != 0 ||
      (reinterpret_cast<uintptr_t>(out) & 3) != 0 || (reinterpret_cast<uintptr_t>(w) & 15) != 0 || (ldw & 15) != 0 ||
      ldw < 64 || pixels < 1) {
    set_error("conv_smallk: unsupported geometry k=%d oc=%d", k_true, g.out_c);
    return MI_PARAM_INVALID;
  }
  const int64_t waves = (pixels + 31) / 32;
  const int blocks = (int)((waves + 3) / 4);
  const int ocb = (g.out_c + 31) / 32, ksteps = (k_true + 31) / 32;
#define MI_SMALLK(KS, OB)                                                                                       \
  launch_kernel((conv_smallk_kernel<KS, OB>), dim3(blocks), dim3(256), 0, stream, in, g, fill, k_true, w, ldw, \
                rq, out)
  if (ksteps == 1) {
    if (ocb == 1) MI_SMALLK(1, 1);
    else if (ocb == 2) MI_SMALLK(1, 2);
    else if (ocb == 3) MI_SMALLK(1, 3);
    else MI_SMALLK(1, 4);
  } else {
    if (ocb == 1) MI_SMALLK(2, 1);
    else if (ocb == 2) MI_SMALLK(2, 2);
    else if (ocb == 3) MI_SMALLK(2, 3);
    else MI_SMALLK(2, 4);
  }
#undef MI_SMALLK
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

// First-layer convolutions: few input channels, so that one row of the window -- kernel_w * in_c consecutive bytes of an
// image row (dilation_w = 1) -- is at most 32 bytes.  The contraction is laid out row by row of the window, each padded
// to 16 or 32 bytes (PARTS chunks of 16), with zero weights in the padding: a lane's 16 bytes of operand are then one
// 16-byte load from any byte address of the image instead of 16 gathered bytes, and nothing is written in between (the
// im2col buffer of 32 x 224 x 224 x 3, 7x7, is 64 MB).  Out-of-image bytes of a row are a byte range, the same for all
// window rows, merged in with two masks made once per pixel.
// The pixels are the MFMA's row operand: a lane ends up with ONE output channel of 16 pixels per accumulator block, its
// requantisation parameters are loaded once and live in registers, and a 4 x 4 byte transposition across neighbouring
// lanes makes dwords of four channels for the stores.  A wave keeps the weights of its up to 64 channels in registers
// and walks tiles of 32 pixels, fetching the next tile's operand before it requantises the current one.
// Bound at large sizes by the vector ALU (about 160 instructions per tile of 32 pixels x 64 channels, 120 of them the
// requantisation), by the loads, whose 64 unaligned addresses take the address unit about 95 cycles, and by the stores; at small
// ones by the latency of one tile.  The order of tiles over the XCDs and the number of waves change nothing; windows of many
// loads go through LDS (conv_window.hip).  us per launch with masks and branches in every tile and divisions by the vector
// ALU (461 instructions) / plain tiles (230) / with the requantisation and stores of conv_store.h: 32 x 224 x 224 x 3 -> 64, 7x7,
// stride 2 25.4 / 22.6 / 20.5; 32 x 224 x 224 x 3 -> 32, 3x3, stride 2 10.3 / - / 8.7; 16 of those 6.5 / 5.65 / 5.5;
// 16 x 160 x 160 x 3 -> 64, 3x3 14.7 / 12.4 / 10.9; 16 x 224 x 224 x 4 -> 32, 5x5 20 / 16.4 / 14.8.
struct ConvRows {
  const int8_t *in;
  const int8_t *w;  // [out_c padded to 64][32 * KS]
  int in_bytes;
  int in_h, in_w, out_w, out_hw, out_c;
  int stride_h, stride_w, dil_h;
  // (small numbers share words and are shifted out of them: a byte of its own comes by a vector load)
  uint32_t pads, sizes, shifts;
  int pixels;
  uint32_t magic_hw, magic_w;  // quotients by out_hw and out_w: umulhi(2 p, magic) >> shift (see magic31)
  int step;                    // tiles that all workgroups of a channel group do at once
  __host__ __device__ __forceinline__ int pad_u() const { return (int16_t)pads; }
  __host__ __device__ __forceinline__ int pad_l() const { return (int)pads >> 16; }
  __host__ __device__ __forceinline__ int in_c() const { return (int)(sizes & 0xff); }
  __host__ __device__ __forceinline__ int kernel_h() const { return (int)(sizes >> 8 & 0xff); }
  __host__ __device__ __forceinline__ int row_bytes() const { return (int)(sizes >> 16 & 0xff); }  // kernel_w * in_c
  __host__ __device__ __forceinline__ uint32_t fill() const { return sizes >> 24; }
  __host__ __device__ __forceinline__ int shift_hw() const { return (int)(shifts & 0xff); }
  __host__ __device__ __forceinline__ int shift_w() const { return (int)(shifts >> 8 & 0xff); }
  __host__ __device__ __forceinline__ bool streams() const { return (shifts >> 16) != 0; }
  __host__ __device__ __forceinline__ int parts() const { return row_bytes() <= 16 ? 1 : 2; }  // 16-byte chunks per window row
};
static_assert(sizeof(ConvRows) + sizeof(RequantCall) + sizeof(int8_t *) <= kShortArgs, "see launch_args.h");

// A tile's operand straight from the image: lane r (of each half) takes pixel 32 * tile + r.
template <int KS>
struct RowsGather {
  const ConvRows &g;
  int r, h, part, line, last16;  // part: which chunk of a window row this lane holds
  int img, ih0, t0;  // the image, the window's first row, the chunk's first byte in an image row
  // A plain tile, the usual one, has all its windows inside the image and all its loads inside the tensor: the loads then
  // differ by a scalar, and no byte needs replacing (those past a window row meet zero weights).
  bool plain;

  __device__ __forceinline__ RowsGather(const ConvRows &g_, int lane)
      : g(g_), r(lane & 31), h(lane >> 5), part(g_.parts() == 2 ? h : 0), line(g_.in_w * g_.in_c()), last16(g_.in_bytes - 16) {}
  __device__ __forceinline__ int window_row(int s) const { return g.parts() == 2 ? s : 2 * s + h; }
  __device__ __forceinline__ void locate(int tile) {
    const int want = tile * 32 + r, p = want < g.pixels ? want : g.pixels - 1;
    const int b = quotient31(p, g.magic_hw, g.shift_hw()), rem = p - b * g.out_hw;
    const int oh = quotient31(rem, g.magic_w, g.shift_w()), ow = rem - oh * g.out_w;
    img = b * (g.in_h * line);
    ih0 = oh * g.stride_h - g.pad_u();
    t0 = (ow * g.stride_w - g.pad_l()) * g.in_c() + 16 * part;
    const int from = t0 - 16 * part, to_last = (g.parts() == 2 ? KS - 1 : 2 * KS - 1) * g.dil_h;
    plain = __all(ih0 >= 0 && ih0 + to_last < g.in_h && from >= 0 && from + g.row_bytes() <= line &&
                  (uint32_t)img + (uint32_t)(ih0 + to_last) * (uint32_t)line + (uint32_t)t0 <= (uint32_t)last16);
  }
  // Every load is a whole 16 bytes inside the tensor: rows above or below the image are clamped (their bytes are
  // replaced), and an address before its first or behind its last 16 bytes is moved in.
  __device__ __forceinline__ int address(int s) const {
    int kh = window_row(s);
    kh = kh < g.kernel_h() ? kh : g.kernel_h() - 1;
    const int ih = min(max(ih0 + kh * g.dil_h, 0), g.in_h - 1);
    return img + ih * line + t0;
  }
  __device__ __forceinline__ void fetch(v4i (&x)[KS]) const {
    if (plain) {
      const int row_step = g.dil_h * line;
      const uint32_t lane_off = (uint32_t)(img + ih0 * line + t0 + (g.parts() == 2 ? 0 : h * row_step));
      const int8_t *row = g.in;
#pragma unroll
      for (int s = 0; s < KS; ++s, row += g.parts() == 2 ? row_step : 2 * row_step)
        x[s] = *reinterpret_cast<const v4i_any *>(row + lane_off);
      return;
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) x[s] = *reinterpret_cast<const v4i_any *>(g.in + min(max(address(s), 0), last16));
  }
  // what was fetched, as the window sees it
  __device__ __forceinline__ void mend(v4i (&x)[KS]) const {
    if (plain) return;
    if (__any(address(0) < 0 || address(KS - 1) > last16)) {  // a load that was moved in: move its bytes back
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int off = address(s), by = off - min(max(off, 0), last16);
        if (by != 0) {
          unsigned __int128 v = __builtin_bit_cast(unsigned __int128, x[s]);
          v = by <= -16 || by >= 16 ? 0 : (by >= 0 ? v >> (8 * by) : v << (-8 * by));
          x[s] = __builtin_bit_cast(v4i, v);
        }
      }
    }
    const uint32_t fill4 = g.fill() * 0x01010101u;
    uint32_t in_row[4];
    row_mask(t0, line, in_row);
    const bool rows_inside = ih0 >= 0 && ih0 + (g.kernel_h() - 1) * g.dil_h < g.in_h;
    if (__all(rows_inside)) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int d = 0; d < 4; ++d) x[s][d] = (int)(((uint32_t)x[s][d] & in_row[d]) | (fill4 & ~in_row[d]));
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bool row_ok = (unsigned)(ih0 + window_row(s) * g.dil_h) < (unsigned)g.in_h;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t m = row_ok ? in_row[d] : 0u;
          x[s][d] = (int)(((uint32_t)x[s][d] & m) | (fill4 & ~m));
        }
      }
    }
  }
  // of 16 bytes that start at byte t of an image row, those inside the row, [-t, line - t); the others are fill
  static __device__ __forceinline__ void row_mask(int t, int line, uint32_t (&m)[4]) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int a = min(max(-t - 4 * d, 0), 4), b = min(max(line - t - 4 * d, 0), 4);
      m[d] = (uint32_t)((((uint64_t)1 << (8 * b)) - 1) & ~(((uint64_t)1 << (8 * a)) - 1));
    }
  }
};

// A tile's accumulators -> bytes in memory (see conv_store.h).
template <int OCB, RequantForm FORM>
struct RowsStore {
  ChannelRequant<OCB, FORM> requant;
  int my_n, my_p;
  uint32_t out_off;

  __device__ __forceinline__ RowsStore(const ConvRows &g, const RequantParams &rq, int n0, int lane) : requant(rq, n0, lane) {
    my_n = n0 + column_channel(OCB, 0, lane & 31 & ~3), my_p = 4 * (lane >> 5) + (lane & 3);
    out_off = (uint32_t)(my_p * g.out_c + my_n);
  }
  __device__ __forceinline__ void store(const ConvRows &g, const RequantParams &rq, v16i (&acc)[OCB], const v16i &sums, int tile,
                                        int n0, int8_t *out) const {
    wait_for_products(acc);
    int8_t *tile_out = out + (int64_t)tile * 32 * g.out_c;
    // (no branch between the pieces of a whole tile: one's chain of dependent instructions fills the gaps of the next)
    requant.in_form(tile * 32 + 32 <= g.pixels, n0, my_n, g.out_c, g.streams(), [&](auto kind, auto streamed) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        // (the transposition needs every lane: those whose pixel is not there store none of their channels)
        requant.template store<decltype(kind)::value, decltype(streamed)::value>(
            rq, acc, sums, q, tile_out + 8 * q * g.out_c + out_off, tile * 32 + 8 * q + my_p < g.pixels ? g.out_c - my_n : 0);
    });
  }
};

// this lane's weights, as the matrix operand of channel block ob and step s
template <int KS, int OCB>
__device__ __forceinline__ void rows_weights(const ConvRows &g, int n0, int lane, v4i (&wf)[OCB][KS]) {
#pragma unroll
  for (int ob = 0; ob < OCB; ++ob)
#pragma unroll
    for (int s = 0; s < KS; ++s)
      wf[ob][s] = *reinterpret_cast<const v4i *>(g.w + (n0 + column_channel(OCB, ob, lane & 31)) * (32 * KS) + 32 * s + 16 * (lane >> 5));
}

// waves per SIMD: three where the weights leave registers for it
constexpr int rows_occupancy(int ks, int ocb, RequantForm form) { return form != kGeneralForm && ks * ocb <= 8 ? 3 : 2; }

template <int KS, int OCB, RequantForm FORM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(rows_occupancy(KS, OCB, FORM)))) void conv_rows_kernel(
    ConvRows g, RequantCall call, int8_t *__restrict__ out) {
  call.load_now();
  asm volatile("" ::"s"(g.in), "s"(g.w), "s"(g.in_bytes), "s"(g.in_h), "s"(g.in_w), "s"(g.out_w), "s"(g.out_hw), "s"(g.out_c), "s"(g.stride_h),
               "s"(g.stride_w), "s"(g.dil_h), "s"(g.pads), "s"(g.sizes), "s"(g.shifts), "s"(g.pixels), "s"(g.magic_hw), "s"(g.magic_w),
               "s"(g.step), "s"(out));
  const RequantParams rq = call.open(g.out_c);
  const int lane = threadIdx.x & 63;
  const int n0 = blockIdx.y * (32 * OCB);
  const int tiles = (g.pixels + 31) >> 5, step = g.step;
  int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= tiles) return;

  v4i wf[OCB][KS];
  rows_weights(g, n0, lane, wf);
  const RowsStore<OCB, FORM> store(g, rq, n0, lane);
  RowsGather<KS> in(g, lane);
  v16i start;
#pragma unroll
  for (int e = 0; e < 16; ++e) start[e] = (int)kAccBias;
  if (FORM != kGeneralForm) asm volatile("" : "+v"(start));  // one block of registers for every tile's first products
  in.locate(tile);
  v4i x[KS];
  in.fetch(x);
  for (; tile < tiles; tile += step) {
    in.mend(x);
    v16i acc[OCB], sums;
#pragma unroll
    for (int e = 0; e < 16; ++e) sums[e] = 0;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int ob = 0; ob < OCB; ++ob)
        acc[ob] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[s], wf[ob][s], s == 0 ? start : acc[ob], 0, 0, 0);
    if (FORM == kGeneralForm && rq.has_zw) {  // the pixels' input sums, in the accumulators' layout: against ones where a window byte is
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        v4i one;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int b = in.window_row(s) < g.kernel_h() ? min(max(g.row_bytes() - 16 * in.part - 4 * d, 0), 4) : 0;
          one[d] = (int)(0x01010101u & (uint32_t)(((uint64_t)1 << (8 * b)) - 1));
        }
        sums = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[s], one, sums, 0, 0, 0);
      }
    }
    if (tile + step < tiles) {  // (wave-uniform)
      in.locate(tile + step);
      in.fetch(x);
    }
    store.store(g, rq, acc, sums, tile, n0, out);
  }
}

bool conv_rows_supported(const ConvGeom &g) {
  const int row = g.kernel_w * g.in_c, parts = row <= 16 ? 1 : 2;
  const int64_t bytes = (int64_t)g.batch * g.in_h * g.in_w * g.in_c;
  return (g.in_c & 15) != 0 && g.dilation_w == 1 && row <= 32 && (g.kernel_h * parts + 1) / 2 <= kConvRowsSteps &&
         bytes >= 16 && bytes < (int64_t)1 << 31 && g.pad_u == (int16_t)g.pad_u && g.pad_l == (int16_t)g.pad_l;
}

// Weights [oc][kh][kw][ic] -> [oc padded to 64][steps of 32 bytes], see ConvRows.
std::vector<int8_t> conv_rows_weights(const int8_t *w, int oc, int kernel_h, int kernel_w, int in_c) {
  const int row = kernel_w * in_c, parts = row <= 16 ? 1 : 2, bytes = 32 * ((kernel_h * parts + 1) / 2);
  std::vector<int8_t> out((size_t)round_up(oc, 64) * bytes, 0);
  for (int c = 0; c < oc; ++c)
    for (int kh = 0; kh < kernel_h; ++kh)
      memcpy(&out[(size_t)c * bytes + (size_t)kh * parts * 16], w + ((size_t)c * kernel_h + kh) * row, (size_t)row);
  return out;
}

int launch_conv_rows(const int8_t *in, const ConvGeom &g, int fill, const int8_t *w, const RequantParams &rq, int8_t *out,
                     hipStream_t stream) {
  ConvRows c{};
  c.in = in;
  c.in_bytes = g.batch * g.in_h * g.in_w * g.in_c;
  c.in_h = g.in_h, c.in_w = g.in_w;
  c.out_w = g.out_w, c.out_hw = g.out_h * g.out_w, c.out_c = g.out_c;
  c.stride_h = g.stride_h, c.stride_w = g.stride_w, c.dil_h = g.dilation_h;
  c.pads = (uint32_t)(uint16_t)g.pad_u | (uint32_t)g.pad_l << 16;
  c.sizes = (uint32_t)g.in_c | (uint32_t)g.kernel_h << 8 | (uint32_t)(g.kernel_w * g.in_c) << 16 | (uint32_t)(uint8_t)fill << 24;
  const int64_t pixels = (int64_t)g.batch * g.out_h * g.out_w;
  c.pixels = (int)pixels;
  c.w = w;
  const int ks = (c.kernel_h() * c.parts() + 1) / 2;
  if (!conv_rows_supported(g) || pixels < 1 || pixels > 0x7fffffff - 4096) {
    set_error("conv_rows: unsupported geometry ic=%d kernel %dx%d", g.in_c, g.kernel_h, g.kernel_w);
    return MI_PARAM_INVALID;
  }
  const int64_t wgs = (pixels + 127) / 128;
  const bool two = g.out_c > 32;
  const bool streams = conv_streams(pixels, g.out_c, two ? 2 : 1);
  const RequantForm form = requant_form(rq);
  const int gy = (g.out_c + (two ? 63 : 31)) / (two ? 64 : 32);
  // as many workgroups as the registers let the device hold, so that a wave walks several tiles on one set of weights.  us at
  // 32 x 224 x 224 x 3 -> 64, 7x7 (two per SIMD): 512 workgroups 22.6, 768 25.4; 16 x 224 x 224 x 3 -> 32, 3x3 (three):
  // 512 5.95, 768 5.65
  const int most = 256 * rows_occupancy(ks, two ? 2 : 1, form);
  const dim3 grid((unsigned)(wgs < most ? wgs : most), (unsigned)gy);
  int shift_hw, shift_w;
  magic31(c.out_hw, &c.magic_hw, &shift_hw);
  magic31(c.out_w, &c.magic_w, &shift_w);
  c.shifts = (uint32_t)shift_hw | (uint32_t)shift_w << 8 | (streams ? 1u << 16 : 0u);
  c.step = 4 * (int)grid.x;
#define MI_ROWS_FORM(KS, FORM)                                                                              \
  if (two) launch_kernel((conv_rows_kernel<KS, 2, FORM>), grid, dim3(256), 0, stream, c, RequantCall::of(rq), out);      \
  else launch_kernel((conv_rows_kernel<KS, 1, FORM>), grid, dim3(256), 0, stream, c, RequantCall::of(rq), out)
#define MI_ROWS(KS)                     \
  case KS:                              \
    if (form == kReluForm) {            \
      MI_ROWS_FORM(KS, kReluForm);      \
    } else if (form == kCarryForm) {    \
      MI_ROWS_FORM(KS, kCarryForm);     \
    } else {                            \
      MI_ROWS_FORM(KS, kGeneralForm);   \
    }                                   \
    break
  switch (ks) {
    MI_ROWS(1);
    MI_ROWS(2);
    MI_ROWS(3);
    MI_ROWS(4);
    MI_ROWS(5);
    MI_ROWS(6);
    MI_ROWS(7);
    MI_ROWS(8);
  }
#undef MI_ROWS
#undef MI_ROWS_FORM
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

// Stride-1 depthwise convolutions with a 3x3 or 5x5 window, int8 weights (no weight zero point) and C % 4 == 0.
// A thread computes four channels of a tile of 4 x OT output pixels.  The byte products are taken four at a time along
// the window row with v_dot4: the dwords of neighbouring pixels (four channels each) are transposed so that a dword holds
// four neighbouring pixels of ONE channel, and an output at an odd position takes the window that starts one pixel before
// it, against weights moved up by one byte.  An image row is fetched and transposed once for the up to KS output rows it
// belongs to.  Accumulators start from kAccBias and are requantised with one 64-bit multiply-add (RequantParams::fast2).
// Bound by the vector ALU at large sizes (3x3: about 10 instructions per output, half of them the requantisation; one
// multiply per product and an unpacking instruction for each operand took about 30), by latency at one image.  us per launch,
// conv_dw16_kernel below -> one form of requantisation and store -> now: 3x3, 16 x 112 x 112 x 192 70.1 -> 23.4 -> 21.9 (3.5 TB/s), on 128
// channels - -> 16.2 -> 14.1, 8 x 115 x 115 x 240 - -> 16.1 -> 14.6, 32 x 56 x 56 x 144 - -> 11.5 -> 10.3, one image of 112 x 112 x 192
// 8.6 -> 4.3 -> 4.2; 5x5, 4 x 80 x 80 x 72 16.4 -> 6.0, 1 x 64 x 64 x 64 7.1 -> 4.1.
struct ConvDwRows {
  const int8_t *in;
  const int32_t *w;    // [KS * (KS == 3 ? 1 : 3)][C]: bytes w0..w2 0 of a window row; 5x5: w0..w3, w4 0 0 0, w3 w4 0 0
  const int32_t *par;  // [5][C]: mult2, c2lo, c2hi, pre, shift
  int8_t *out;
  int in_h, in_w, ch, out_h, out_w, pad_u, pad_l;
  int groups, strips, bands;  // channels / 4, output columns / 4, output rows / OT, rounded up
  int total;                  // batch * bands * strips * groups
  int zsplat, amin, amax;
  uint32_t magic_groups, magic_strips, magic_bands, shifts;  // quotients by those (see magic31), shifts a byte each
  void set_quotients() {
    int s[3];
    magic31(groups, &magic_groups, s);
    magic31(strips, &magic_strips, s + 1);
    magic31(bands, &magic_bands, s + 2);
    shifts = (uint32_t)(s[0] | s[1] << 8 | s[2] << 16);
  }
};
static_assert(sizeof(ConvDwRows) <= kShortArgs, "see launch_args.h");

// Outputs of up to kStreamedMost bytes are stored non-temporally (STREAMED) from this many channels, where a pixel's are at least a
// line; half as many bytes where pixels begin inside a line's 32-byte sectors, which two stores then share.  us, temporal -> streamed:
// 16 x 112 x 112 on 128 channels 15.9 -> 14.3, 32 x 56 x 56 on 144 11.4 -> 11.1, 8 x 80 x 80 on 72, 5x5 6.9 -> 7.4; 32 x 112 x 112 on 192
// (77 MB) 43.8 -> 45.7; 12 x 112 x 112 on 128 (19 MB) 11.9 -> 10.5, on 160 13.6 -> 12.9, on 140 13.4 -> 14.1; 16 x 57 x 57 (7 MB) on 140 even,
// on 200 8.9 -> 8.4.
constexpr int kDwStreamedLeast = 128;

// RELU: no output is below the zero point.  The rounding's sign term is then a constant (as in kReluForm of conv_store.h).  us:
// 16 x 112 x 112 on 128 channels 15.9 -> 15.1, 32 x 56 x 56 on 144 11.4 -> 10.5, 8 x 80 x 80 on 72, 5x5 6.95 -> 6.75.
// A launch lasts a few times its way to the first input: 165 instructions with three divisions and two scalar round trips, now 110 and one.
// us: 1 x 112 x 112 x 192 3.92 -> 3.71, 8 x 128 x 128 x 96 9.72 -> 9.53, 16 x 112 x 112 x 192 19.75 -> 19.15, 2 x 66 x 66 x 128 3.32 -> 3.16.
template <int KS, int OT, bool RELU, bool STREAMED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void conv_dw_rows_kernel(ConvDwRows g) {
  constexpr int PX = KS + 3;       // input pixels per row of four outputs
  constexpr int WR = KS == 3 ? 1 : 3;  // weight dwords per channel and window row
  asm volatile("" ::"s"(g.in), "s"(g.w), "s"(g.par), "s"(g.out), "s"(g.in_h), "s"(g.in_w), "s"(g.ch), "s"(g.out_h), "s"(g.out_w), "s"(g.pad_u),
               "s"(g.pad_l), "s"(g.groups), "s"(g.strips), "s"(g.bands), "s"(g.total), "s"(g.zsplat), "s"(g.amin), "s"(g.amax),
               "s"(g.magic_groups), "s"(g.magic_strips), "s"(g.magic_bands), "s"(g.shifts));
  // as below: workgroups that share an XCD get one contiguous band of the output
  int bid = blockIdx.x;
  const int per = ((g.total + 255) >> 8) >> 3;  // an eighth of the grid
  if (bid < per * 8) bid = (bid & 7) * per + (bid >> 3);
  const int idx = bid * 256 + threadIdx.x;
  if (idx >= g.total) return;
  const int rest = quotient31(idx, g.magic_groups, g.shifts & 0xff), c0 = (idx - rest * g.groups) * 4;
  const int up = quotient31(rest, g.magic_strips, g.shifts >> 8 & 0xff), ow0 = (rest - up * g.strips) * 4;
  const int b = quotient31(up, g.magic_bands, g.shifts >> 16), oh0 = (up - b * g.bands) * OT;
  const int ih0 = oh0 - g.pad_u, iw0 = ow0 - g.pad_l;
  const int line = g.in_w * g.ch;

  uint32_t px[OT + KS - 1][PX];
  const int8_t *img = g.in + (int64_t)b * g.in_h * line + c0;
  const bool inside = ih0 >= 0 && iw0 >= 0 && ih0 + OT + KS - 2 < g.in_h && iw0 + PX <= g.in_w;
  if (__all(inside)) {
    const int8_t *row = img + (int64_t)ih0 * line + iw0 * g.ch;
#pragma unroll
    for (int i = 0; i < OT + KS - 1; ++i)
#pragma unroll
      for (int j = 0; j < PX; ++j) px[i][j] = *reinterpret_cast<const uint32_t *>(row + i * line + j * g.ch);
  } else {  // (every load is inside the tensor; what lies outside the image is replaced by the input zero point)
#pragma unroll
    for (int i = 0; i < OT + KS - 1; ++i) {
      const int ih = ih0 + i, ihc = min(max(ih, 0), g.in_h - 1);
#pragma unroll
      for (int j = 0; j < PX; ++j) {
        const int iw = iw0 + j, iwc = min(max(iw, 0), g.in_w - 1);
        px[i][j] = *reinterpret_cast<const uint32_t *>(img + ihc * line + iwc * g.ch);
      }
    }
#pragma unroll
    for (int i = 0; i < OT + KS - 1; ++i)
#pragma unroll
      for (int j = 0; j < PX; ++j)
        if (ih0 + i != min(max(ih0 + i, 0), g.in_h - 1) || iw0 + j != min(max(iw0 + j, 0), g.in_w - 1))
          px[i][j] = (uint32_t)g.zsplat;
  }

  v4i acc[OT][4];  // [row][column], four channels
#pragma unroll
  for (int o = 0; o < OT; ++o)
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[o][x][c] = (int)kAccBias;
  v4i w[KS][WR];
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int p = 0; p < WR; ++p) w[k][p] = *reinterpret_cast<const v4i *>(g.w + (int64_t)(k * WR + p) * g.ch + c0);
  v4i par[5];
#pragma unroll
  for (int a = 0; a < 5; ++a) par[a] = *reinterpret_cast<const v4i *>(g.par + (int64_t)a * g.ch + c0);
  if (RELU) par[2] = par[2] + par[3] + 1;  // see kReluForm

#pragma unroll
  for (int i = 0; i < OT + KS - 1; ++i) {
    uint32_t lo[PX / 2], hi[PX / 2];  // pixel pairs: bytes a0 b0 a1 b1 / a2 b2 a3 b3
#pragma unroll
    for (int t = 0; t < PX / 2; ++t) {
      lo[t] = __builtin_amdgcn_perm(px[i][2 * t + 1], px[i][2 * t], 0x05010400u);
      hi[t] = __builtin_amdgcn_perm(px[i][2 * t + 1], px[i][2 * t], 0x07030602u);
    }
    int win[PX / 2 - 1][4];  // [first pixel / 2][channel]: four pixels of a channel
#pragma unroll
    for (int t = 0; t < PX / 2 - 1; ++t) {
      win[t][0] = (int)__builtin_amdgcn_perm(lo[t + 1], lo[t], 0x05040100u);
      win[t][1] = (int)__builtin_amdgcn_perm(lo[t + 1], lo[t], 0x07060302u);
      win[t][2] = (int)__builtin_amdgcn_perm(hi[t + 1], hi[t], 0x05040100u);
      win[t][3] = (int)__builtin_amdgcn_perm(hi[t + 1], hi[t], 0x07060302u);
    }
#pragma unroll
    for (int o = 0; o < OT; ++o) {
      const int k = i - o;
      if (k < 0 || k >= KS) continue;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int w0 = w[k][0][c], w1 = (int)((uint32_t)w0 << 8);
        acc[o][0][c] = __builtin_amdgcn_sdot4(win[0][c], w0, acc[o][0][c], false);
        acc[o][1][c] = __builtin_amdgcn_sdot4(win[0][c], w1, acc[o][1][c], false);
        acc[o][2][c] = __builtin_amdgcn_sdot4(win[1][c], w0, acc[o][2][c], false);
        acc[o][3][c] = __builtin_amdgcn_sdot4(win[1][c], w1, acc[o][3][c], false);
        if constexpr (KS == 5) {  // the window's last pixels: columns 4..7 hold what the first windows left out
          const int e = w[k][1][c], d = w[k][2][c];
          acc[o][0][c] = __builtin_amdgcn_sdot4(win[2][c], e, acc[o][0][c], false);
          acc[o][1][c] = __builtin_amdgcn_sdot4(win[2][c], d, acc[o][1][c], false);
          acc[o][2][c] = __builtin_amdgcn_sdot4(win[2][c], (int)((uint32_t)e << 16), acc[o][2][c], false);
          acc[o][3][c] = __builtin_amdgcn_sdot4(win[2][c], (int)((uint32_t)d << 16), acc[o][3][c], false);
        }
      }
    }
  }

  int amin_v = g.amin, amax_v = g.amax;
  asm volatile("" : "+v"(amin_v), "+v"(amax_v));  // kept in vector registers, as v_med3 wants them
  // (a dot product's result needs three wait states before another instruction reads it; the compiler keeps them, but not
  //  where that instruction is inline assembly)
#pragma unroll
  for (int o = 0; o < OT; ++o) asm volatile("s_nop 3" : "+v"(acc[o][0]), "+v"(acc[o][1]), "+v"(acc[o][2]), "+v"(acc[o][3]));
  int8_t *dst = g.out + (((int64_t)b * g.out_h + oh0) * g.out_w + ow0) * g.ch + c0;
#pragma unroll
  for (int o = 0; o < OT; ++o)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      int y[4];
      int32_t t[4];
      if (RELU) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint64_t c2 = (uint64_t)(uint32_t)par[2][c] << 32 | (uint32_t)par[1][c];
          t[c] = (int32_t)(((uint64_t)(uint32_t)acc[o][x][c] * (uint32_t)par[0][c] + c2) >> 32);
        }
      } else {
        uint64_t p2[4], carry[4], unused;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint64_t c2 = (uint64_t)(uint32_t)par[2][c] << 32 | (uint32_t)par[1][c];
          asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=&v"(p2[c]), "=s"(carry[c]) : "v"(acc[o][x][c]), "v"(par[0][c]), "v"(c2));
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
          asm("v_addc_co_u32_e64 %0, %1, %2, %3, %4"
              : "=v"(t[c]), "=s"(unused)
              : "v"((int32_t)(p2[c] >> 32)), "v"(par[3][c]), "s"(carry[c]));
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        t[c] >>= par[4][c];
        asm("v_med3_i32 %0, %1, %2, %3" : "=v"(y[c]) : "v"(t[c]), "v"(amin_v), "v"(amax_v));
      }
      const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)y[1], (uint32_t)y[0], 0x0c0c0400u);
      const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)y[3], (uint32_t)y[2], 0x0c0c0400u);
      if (oh0 + o < g.out_h && ow0 + x < g.out_w) {
        const uint32_t four = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
        uint32_t *to = reinterpret_cast<uint32_t *>(dst + ((int64_t)o * g.out_w + x) * g.ch);
        if (STREAMED) {
          __builtin_nontemporal_store(four, to);
        } else {
          *to = four;
        }
      }
    }
}

bool conv_dw_rows_supported(const ConvGeom &g) {
  return (g.kernel_h == 3 || g.kernel_h == 5) && g.kernel_w == g.kernel_h && g.stride_h == 1 && g.stride_w == 1 &&
         g.dilation_h == 1 && g.dilation_w == 1 && (g.out_c & 3) == 0 &&
         (int64_t)g.in_h * g.in_w * g.out_c < (int64_t)1 << 31 &&
         (int64_t)g.batch * g.out_h * ((g.out_w + 3) / 4) * (g.out_c / 4) < ((int64_t)1 << 31) - 256;
}

// Weights [C][KS][KS] -> the dwords of ConvDwRows::w.
std::vector<int32_t> conv_dw_rows_weights(const int8_t *w, int ch, int ks) {
  const int wr = ks == 3 ? 1 : 3;
  std::vector<int32_t> out((size_t)ks * wr * ch);
  for (int c = 0; c < ch; ++c)
    for (int k = 0; k < ks; ++k) {
      const int8_t *row = w + ((size_t)c * ks + k) * ks;
      uint8_t d[3][4] = {};
      for (int i = 0; i < (ks < 4 ? ks : 4); ++i) d[0][i] = (uint8_t)row[i];
      if (ks == 5) d[1][0] = (uint8_t)row[4], d[2][0] = (uint8_t)row[3], d[2][1] = (uint8_t)row[4];
      for (int p = 0; p < wr; ++p) memcpy(&out[(size_t)(k * wr + p) * ch + c], d[p], 4);
    }
  return out;
}

template <int KS, int OT>
static int launch_dw_rows(ConvDwRows c, int batch, int zo, hipStream_t stream) {
  c.bands = (c.out_h + OT - 1) / OT;
  c.total = batch * c.bands * c.strips * c.groups;
  c.set_quotients();
  const bool streamed = c.ch >= kDwStreamedLeast &&
                        (int64_t)batch * c.out_h * c.out_w * c.ch <= (c.ch % 32 == 0 ? kStreamedMost : kStreamedMost / 2);
  const auto kernel = c.amin >= zo ? (streamed ? conv_dw_rows_kernel<KS, OT, true, true> : conv_dw_rows_kernel<KS, OT, true, false>)
                                   : (streamed ? conv_dw_rows_kernel<KS, OT, false, true> : conv_dw_rows_kernel<KS, OT, false, false>);
  launch_kernel(kernel, dim3((c.total + 255) / 256), dim3(256), 0, stream, c);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

int launch_conv_dw_rows(const int8_t *in, const ConvGeom &g, const int32_t *w, const int32_t *par, int zx8, int zo, int amin,
                        int amax, int8_t *out, hipStream_t stream) {
  if (!conv_dw_rows_supported(g) || ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 3) != 0) {
    set_error("conv_dw_rows: unsupported geometry");
    return MI_PARAM_INVALID;
  }
  ConvDwRows c{in,      w,       par,     out,     g.in_h,      g.in_w, g.out_c, g.out_h, g.out_w,
               g.pad_u, g.pad_l, g.out_c / 4, (g.out_w + 3) / 4, 0,      0,       (zx8 & 0xff) * 0x01010101, amin, amax};
  // Tall tiles fetch and transpose fewer rows twice, flat ones make more threads.  us at one / two / four / eight rows: 3x3,
  // 1 x 112 x 112 x 192 4.8, 5.3, 5.5, 7.6; 8 x 115 x 115 x 240 20.3, 17.8, 17.1, 19.6; 16 x 112 x 112 x 192 28.2, 23.5, 22.1,
  // 23.8; 5x5, 1 x 64 x 64 x 64 4.1, 4.9, 6.4; 4 x 80 x 80 x 72 6.4, 6.0, 7.6.
  const int64_t flat = (int64_t)g.batch * g.out_h * c.strips * c.groups;  // threads at one row each
  if (g.kernel_h == 3) {
    if (flat >= 1 << 20) return launch_dw_rows<3, 4>(c, g.batch, zo, stream);
    if (flat >= 1 << 18) return launch_dw_rows<3, 2>(c, g.batch, zo, stream);
    return launch_dw_rows<3, 1>(c, g.batch, zo, stream);
  }
  if (flat >= 1 << 16) return launch_dw_rows<5, 2>(c, g.batch, zo, stream);
  return launch_dw_rows<5, 1>(c, g.batch, zo, stream);
}

__global__ __launch_bounds__(256) void conv_dw_kernel(const int8_t *__restrict__ in, ConvGeom g,
                                                      const int16_t *__restrict__ w16,
                                                      const int32_t *__restrict__ bias, int zx8, RequantParams rq,
                                                      int8_t *__restrict__ out) {
  const int ch = g.out_c, n_pad = padded_channels(ch);
  const int64_t total = (int64_t)g.batch * g.out_h * g.out_w * ch;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = idx / ch;
    const int c = (int)(idx - p * ch);
    const int b = (int)(p / ((int64_t)g.out_h * g.out_w));
    const int rem = (int)(p - (int64_t)b * g.out_h * g.out_w);
    const int oh = rem / g.out_w, ow = rem - oh * g.out_w;
    const int8_t *img = in + (int64_t)b * g.in_h * g.in_w * ch;
    uint32_t acc = (uint32_t)bias[c];
    for (int kh = 0; kh < g.kernel_h; ++kh) {
      const int ih = oh * g.stride_h - g.pad_u + kh * g.dilation_h;
      if (ih < 0 || ih >= g.in_h) continue;
      for (int kw = 0; kw < g.kernel_w; ++kw) {
        const int iw = ow * g.stride_w - g.pad_l + kw * g.dilation_w;
        if (iw < 0 || iw >= g.in_w) continue;
        const int16_t xv = (int16_t)((int)img[((int64_t)ih * g.in_w + iw) * ch + c] - zx8);
        const int16_t wv = w16[(kh * g.kernel_w + kw) * ch + c];
        acc += (uint32_t)((int32_t)xv * (int32_t)wv);
      }
    }
    const int32_t mult = rq.mult(n_pad)[c], e = rq.rshift[c], ls = rq.lshift(n_pad)[c];
    int32_t y = rdiv_pot(srdhm((int32_t)(acc << ls), mult), e);
    y = (int32_t)((uint32_t)y + (uint32_t)rq.zo);
    y = y > rq.amin ? y : rq.amin;  // MSMAX first, then MSMIN (conv_depthwise_int8.c:49-50)
    y = y < rq.amax ? y : rq.amax;
    out[idx] = (int8_t)y;
  }
}

// Channel-vectorised variant for C % 8 == 0: one thread produces CG = 16 (or 8, when C is not a multiple of 16)
// consecutive channels of one output pixel, so every tap is one CG-byte activation load and 2 * CG bytes of weights,
// and the store is one CG-byte row segment.
// A tap outside the image reads as the input zero point (the matching -zx * w is already in bias_folded), so the
// inner product is sum_t x_t * w_t with no subtraction.  TAPS > 0 (kernel_h * kernel_w known at compile time): the
// loads of all taps are issued before the first multiply.  TAPS == 0: any kernel size, five taps per batch of loads.  FAST: the host
// proved the cheap rounding form exact for every channel (no left shifts to fetch).
// A thread reads the parameters of its CG channels from arrays, four channels a load: with RequantChannel, a load of 16 bytes per
// channel, every channel of a wave's lines was fetched on its own.  us, records -> arrays: 3x3 at stride 2, 4 x 151 x 151 x 96
// 14.1 -> 8.15, 16 x 135 x 135 x 128 30.6 -> 20.7; 32 x 50 x 50 x 72 with left shifts 29.7 -> 14.2; 7x7, 16 x 39 x 39 x 960 197 -> 140,
// 1 x 30 x 30 x 72 12.9 -> 11.4.
template <int TAPS, int CG, bool FAST>
__global__ __launch_bounds__(256) void conv_dw16_kernel(const int8_t *__restrict__ in, ConvGeom g,
                                                        const int16_t *__restrict__ w16,
                                                        const int32_t *__restrict__ bias_folded, int zx8,
                                                        RequantParams rq, int8_t *__restrict__ out) {
  static_assert(CG == 8 || CG == 16, "channels per thread");
  constexpr int XW = CG / 4;  // dwords of activations per tap
  constexpr int WQ = CG / 8;  // 16-byte vectors of int16 weights per tap
  const int ch = g.out_c, groups = ch / CG, n_pad = padded_channels(ch);
  const int64_t total = (int64_t)g.batch * g.out_h * g.out_w * groups;
  const int zsplat = (zx8 & 0xff) * 0x01010101;
  union XV {
    int32_t d[XW];
    int8_t b[CG];
  };
  union WV {
    v4i v[WQ];
    int16_t h[CG];
  };
  auto load_x = [](const int8_t *p, XV *x) {
    if constexpr (CG == 16) {
      const v4i v = *reinterpret_cast<const v4i *>(p);
      x->d[0] = v.x, x->d[1] = v.y, x->d[2] = v.z, x->d[3] = v.w;
    } else {
      const v2i v = *reinterpret_cast<const v2i *>(p);
      x->d[0] = v.x, x->d[1] = v.y;
    }
  };
  // Consecutive workgroup ids are dealt round-robin over the 8 XCDs, each with an L2 of its own; a 3x3 window reads
  // three image rows, so with ids in pixel order every XCD would fetch nearly the whole image (measured: 8.0 MB for
  // a 2.4 MB image).  Ids that share an XCD are mapped to one contiguous band of the output instead.
  int64_t bid = blockIdx.x;
  {
    const int64_t per = gridDim.x >> 3;
    if (bid < per * 8) bid = (bid & 7) * per + (bid >> 3);
  }
  for (int64_t idx = bid * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = idx / groups;
    const int c0 = (int)(idx - p * groups) * CG;
    const int b = (int)(p / ((int64_t)g.out_h * g.out_w));
    const int rem = (int)(p - (int64_t)b * g.out_h * g.out_w);
    const int oh = rem / g.out_w, ow = rem - oh * g.out_w;
    const int8_t *img = in + (int64_t)b * g.in_h * g.in_w * ch + c0;
    uint32_t acc[CG];
    {
      const v4i *bp = reinterpret_cast<const v4i *>(bias_folded + c0);
#pragma unroll
      for (int q = 0; q < CG / 4; ++q) {
        const v4i bv = bp[q];
        acc[4 * q + 0] = (uint32_t)bv.x;
        acc[4 * q + 1] = (uint32_t)bv.y;
        acc[4 * q + 2] = (uint32_t)bv.z;
        acc[4 * q + 3] = (uint32_t)bv.w;
      }
    }
    auto mac = [&](XV xv, const WV &wv, bool inside) {
#pragma unroll
      for (int q = 0; q < XW; ++q) xv.d[q] = inside ? xv.d[q] : zsplat;
#pragma unroll
      for (int j = 0; j < CG; ++j) acc[j] += (uint32_t)((int32_t)xv.b[j] * (int32_t)wv.h[j]);  // 8 bit x 10 bit
    };
    auto tap_address = [&](int kh, int kw, bool *inside) -> const int8_t * {
      const int ih = oh * g.stride_h - g.pad_u + kh * g.dilation_h;
      const int iw = ow * g.stride_w - g.pad_l + kw * g.dilation_w;
      *inside = ih >= 0 && ih < g.in_h && iw >= 0 && iw < g.in_w;
      const int ihc = ih < 0 ? 0 : (ih >= g.in_h ? g.in_h - 1 : ih);
      const int iwc = iw < 0 ? 0 : (iw >= g.in_w ? g.in_w - 1 : iw);
      return img + ((int64_t)ihc * g.in_w + iwc) * ch;
    };
    if (TAPS > 0) {
      XV xv[TAPS > 0 ? TAPS : 1];
      WV wv[TAPS > 0 ? TAPS : 1];
      bool inside[TAPS > 0 ? TAPS : 1];
#pragma unroll
      for (int t = 0; t < TAPS; ++t) {
        const int kh = t / g.kernel_w, kw = t - kh * g.kernel_w;
        load_x(tap_address(kh, kw, &inside[t]), &xv[t]);
        const v4i *wp = reinterpret_cast<const v4i *>(w16 + (int64_t)t * ch + c0);
#pragma unroll
        for (int q = 0; q < WQ; ++q) wv[t].v[q] = wp[q];
      }
#pragma unroll
      for (int t = 0; t < TAPS; ++t) mac(xv[t], wv[t], inside[t]);
    } else {
      // five taps at a time (a row of a 5x5 kernel): their loads are issued together, so a kernel of T taps costs
      // T / 5 memory round trips instead of T
      constexpr int B = 5;
      const int taps = g.kernel_h * g.kernel_w;
      int kh = 0, kw = 0;  // of tap t0 + u, kept by stepping (no division per tap)
      for (int t0 = 0; t0 < taps; t0 += B) {
        XV xv[B];
        WV wv[B];
        bool inside[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const bool past = t0 + u >= taps;  // past the last tap: a re-read of the last one that is not used
          const int t = past ? taps - 1 : t0 + u;
          load_x(tap_address(past ? g.kernel_h - 1 : kh, past ? g.kernel_w - 1 : kw, &inside[u]), &xv[u]);
          const bool wrap_w = kw + 1 == g.kernel_w;
          kw = wrap_w ? 0 : kw + 1;
          kh = wrap_w ? kh + 1 : kh;
          const v4i *wp = reinterpret_cast<const v4i *>(w16 + (int64_t)t * ch + c0);
#pragma unroll
          for (int q = 0; q < WQ; ++q) wv[u].v[q] = wp[q];
        }
#pragma unroll
        for (int u = 0; u < B; ++u)
          if (t0 + u < taps) mac(xv[u], wv[u], inside[u]);
      }
    }
    union {
      int32_t d[XW];
      int8_t b[CG];
    } o;
#pragma unroll
    for (int q = 0; q < CG / 4; ++q) {
      const v4i m4 = *reinterpret_cast<const v4i *>(rq.mult(n_pad) + c0 + 4 * q);
      const v4i rs4 = *reinterpret_cast<const v4i *>(rq.rshift + c0 + 4 * q);
      v4i ls4 = {0, 0, 0, 0};
      if (!FAST) ls4 = *reinterpret_cast<const v4i *>(rq.lshift(n_pad) + c0 + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int32_t y;
        if (FAST) {
          y = rdiv_pot_fast(srdhm_nosat((int32_t)acc[4 * q + e], m4[e]), rs4[e], (1 << rs4[e]) >> 1);
        } else {
          y = rdiv_pot(srdhm((int32_t)(acc[4 * q + e] << ls4[e]), m4[e]), rs4[e]);
        }
        y = (int32_t)((uint32_t)y + (uint32_t)rq.zo);
        y = y > rq.amin ? y : rq.amin;  // MSMAX first, then MSMIN (conv_depthwise_int8.c:49-50)
        y = y < rq.amax ? y : rq.amax;
        o.b[4 * q + e] = (int8_t)y;
      }
    }
    if constexpr (CG == 16) {
      *reinterpret_cast<v4i *>(out + p * ch + c0) = v4i{o.d[0], o.d[1], o.d[2], o.d[3]};
    } else {
      *reinterpret_cast<v2i *>(out + p * ch + c0) = v2i{o.d[0], o.d[1]};
    }
  }
}

template <int TAPS, int CG>
static void launch_dw_vec(const int8_t *in, const ConvGeom &g, const int16_t *w16, const int32_t *bias_folded, int zx8,
                          const RequantParams &rq, int8_t *out, hipStream_t stream) {
  const int64_t total = (int64_t)g.batch * g.out_h * g.out_w * (g.out_c / CG);
  const int64_t want = (total + 255) / 256;
  const int blocks = (int)(want < 1 ? 1 : (want > 1048576 ? 1048576 : want));
  if (rq.fast) {
    launch_kernel((conv_dw16_kernel<TAPS, CG, true>), dim3(blocks), dim3(256), 0, stream, in, g, w16, bias_folded,
                  zx8, rq, out);
  } else {
    launch_kernel((conv_dw16_kernel<TAPS, CG, false>), dim3(blocks), dim3(256), 0, stream, in, g, w16, bias_folded,
                  zx8, rq, out);
  }
}

int launch_conv_dw(const int8_t *in, const ConvGeom &g, const int16_t *w16, const int32_t *bias,
                   const int32_t *bias_folded, int zx8, const RequantParams &rq, int8_t *out, hipStream_t stream) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  const bool vec16 = aligned && (g.out_c & 15) == 0, vec8 = aligned && (g.out_c & 7) == 0;
  const bool taps9 = g.kernel_h * g.kernel_w == 9;
  // kernels larger than 3x3 on few pixels: a thread's chain of taps is what the launch lasts, and there are SIMDs to
  // spare, so half the channels per thread
  const bool k5 = g.kernel_h == 5 && g.kernel_w == 5;  // (compile-time taps: 6.4 instead of 7.2 us)
  const bool long_chain = !taps9 && (int64_t)g.batch * g.out_h * g.out_w * (g.out_c >> 4) < 65536;
  if (vec8 && (!vec16 || long_chain)) {  // 8, 24, 40, ... channels
    if (taps9) launch_dw_vec<9, 8>(in, g, w16, bias_folded, zx8, rq, out, stream);
    else if (k5) launch_dw_vec<25, 8>(in, g, w16, bias_folded, zx8, rq, out, stream);
    else launch_dw_vec<0, 8>(in, g, w16, bias_folded, zx8, rq, out, stream);
  } else if (vec16) {
    if (taps9) launch_dw_vec<9, 16>(in, g, w16, bias_folded, zx8, rq, out, stream);
    else launch_dw_vec<0, 16>(in, g, w16, bias_folded, zx8, rq, out, stream);
  } else {
    const int64_t total = (int64_t)g.batch * g.out_h * g.out_w * g.out_c;
    const int64_t want = (total + 255) / 256;
    const int blocks = (int)(want < 1 ? 1 : (want > 1048576 ? 1048576 : want));
    launch_kernel(conv_dw_kernel, dim3(blocks), dim3(256), 0, stream, in, g, w16, bias, zx8, rq, out);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
