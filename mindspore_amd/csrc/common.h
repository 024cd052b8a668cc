// Internal declarations shared by the HIP translation units of libmi355x_int8.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "../../include/mi355x_int8.h"
#include "conv_geom.h"

namespace mi {

void set_error(const char *fmt, ...);

#define MI_HIP_CHECK(expr)                                                                   \
  do {                                                                                       \
    hipError_t _e = (expr);                                                                  \
    if (_e != hipSuccess) {                                                                  \
      mi::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, __LINE__); \
      return MI_ERROR;                                                                       \
    }                                                                                        \
  } while (0)

// For tests (mi_debug_last_kernel): what this thread launched last.
inline thread_local const void *t_last_kernel = nullptr;

// A launch; hipGetLastError says what became of it.  As <<< >>> does it, without its way round a stub that parks the grid in thread-local
// storage and fetches it again: 2.39 -> 2.22 us of the host (empty kernel, 96 bytes of arguments; hipModuleLaunchKernel 2.19).
template <typename T>
struct Given { typedef T type; };
template <typename... P>
inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, typename Given<P>::type... args) {
  void *list[] = {const_cast<void *>(static_cast<const void *>(&args))...};
  t_last_kernel = reinterpret_cast<const void *>(kernel);
  (void)hipLaunchKernel(t_last_kernel, grid, block, list, lds, stream);
}

inline int round_up(int x, int m) { return (x + m - 1) / m * m; }
inline int64_t round_up64(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

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

// Weight rows (output channels) and the contraction dimension are padded so that no kernel needs bounds checks on
// the weight operand: rows to a multiple of kNPad, K to a multiple of kKPad (bytes, two 128-byte GEMM steps), zero filled.
constexpr int kNPad = 256;
constexpr int kKPad = 256;
__host__ __device__ inline int padded_k(int k) { return (k + kKPad - 1) & ~(kKPad - 1); }
__host__ __device__ inline int padded_channels(int n) { return (n + kNPad - 1) & ~(kNPad - 1); }

// The value the 256 x 256 GEMM tile's accumulators start from (taken out again in the epilogue); the host's proof that
// the cheap rounding form cannot overflow includes it.
constexpr uint32_t kAccBias = 0x2AAAAAAAu;

// ---- int8 requantising epilogue parameters (device arrays are padded to kNPad entries) ----
// What the decode kernels, whose waves finish an output per lane, need of a channel, in one load.
struct alignas(16) RequantChannel {
  int32_t mult;     // 31-bit mantissa
  int32_t bias2;    // K*zx*zw - zx*sum(w) + bias
  uint32_t shifts;  // e = -right_shift clamped to [0, 31], and above its byte the left shift (generic path only)
  int32_t zw;       // weight zero point
  __device__ __forceinline__ int32_t rshift() const { return (int32_t)(shifts & 31); }
  __device__ __forceinline__ int32_t lshift() const { return (int32_t)(shifts >> 8); }
};
struct RequantParams {
  const RequantChannel *each;
  const int32_t *rshift, *zw;
  int32_t zo, amin, amax;
  int has_zw;  // any weight zero point is non-zero -> input row sums are needed
  int fast;    // host proved: all lshift == 0, 1 <= e <= 30, no mult == INT32_MIN, amin <= amax, and none of
               // acc + bias2, srdhm + 2^(e-1) + (zo << e) can overflow int32
  // Single-multiply form of the cheap rounding, for accumulators that start from kAccBias (gemm_i8.hip).  With
  // a = accumulator register read as unsigned (true sum + kAccBias [- rowsum * zw]):
  //   x = high dword of (a * mult2 + c2)      == floor(((sum + bias2) * mult + 2^30) / 2^31), the doubling high mul
  //   y = clamp((x + pre + [x >= 0]) >> e)    pre = 2^(e-1) + (zo << e) - 1; [x >= 0] is the carry of a * mult2 + c2
  // mult2 = 2 * mult, c2 = 2 * (bias2 - kAccBias) * mult + 2^31 (mod 2^64, negative as a signed number), in dwords.
  const uint32_t *mult2, *c2lo, *c2hi;
  const int32_t *pre;
  int most_shift;  // the largest e
  int fast2;   // fast, and every mult >= 0, every c2 < 0, and K * 16384 + K * 128 * |zw| <= kAccBias (a in [0, 2^31))

  // The arrays stand one behind the other, of `stride` channels each.  (mult2 to zw are arrays of their own because a wave reads 32
  // to 64 channels of them: with 16 bytes a channel the window convolutions took 5 % longer.)  Behind zw stand arrays of the records'
  // mult, bias2 and lshift, for kernels whose threads read several neighbouring channels: 4 to 16 records a thread are as many
  // scattered loads (conv_dw16_kernel has the figures).
  static constexpr int kWordsPerChannel = 4 + 9;
  __host__ __device__ __forceinline__ const int32_t *mult(int stride) const { return zw + stride; }
  __host__ __device__ __forceinline__ const int32_t *bias2(int stride) const { return zw + 2 * (int64_t)stride; }
  __host__ __device__ __forceinline__ const int32_t *lshift(int stride) const { return zw + 3 * (int64_t)stride; }
  __host__ __device__ __forceinline__ void set_channels(const RequantChannel *block, int stride) {
    each = block;
    mult2 = reinterpret_cast<const uint32_t *>(block + stride);
    c2lo = mult2 + stride;
    c2hi = c2lo + stride;
    pre = reinterpret_cast<const int32_t *>(c2hi + stride);
    rshift = pre + stride;
    zw = rshift + stride;
  }
};

// ---- fp32 dequantising epilogue (dynamic-quant MatMul) ----
struct alignas(16) DequantChannel {  // as RequantChannel
  float wscale;  // (float)filter_scale (per-tensor is broadcast at Prepare)
  int32_t wsum;  // sum_k w[n][k]
  float bias;    // 0 where there is none
  int32_t unused;
};
struct DequantParams {
  const DequantChannel *each;
  const float *wscale, *bias;
  const int32_t *wsum;
  const mi_dq_params *qp_dev;    // input scale / zero point on the device, or nullptr -> use sx / zx below
  float sx;
  int32_t zx;
  int32_t zw0;
  int32_t deep;  // true K
  int32_t act;
  int32_t per_row;  // input scale of row r is qp_dev[r].scale_f; the zero point is qp_dev[0].zero_point
  int32_t has_bias;  // (adding a bias of 0 would turn -0 into 0)

  static constexpr int kWordsPerChannel = 4 + 3;  // the arrays stand as those of RequantParams do
  __host__ __device__ __forceinline__ void set_channels(const DequantChannel *block, int stride) {
    each = block;
    wscale = reinterpret_cast<const float *>(block + stride);
    bias = wscale + stride;
    wsum = reinterpret_cast<const int32_t *>(bias + stride);
  }
};

// Packed weights: n_pad rows (output channels) of k_pad contraction bytes, zero filled past K, with row stride ldw.
// The stride is skewed to an odd multiple of 256 bytes: the kernels fetch 16 rows x 64 bytes per wave instruction,
// and with a power-of-two stride those 16 requests would all fall into the same memory channel.
struct WeightView {
  const int8_t *w;
  int k_pad;
  int ldw;
  // Second copy for the matrix-core decode kernel and the GEMM's K-block loops, or nullptr: the same bytes regrouped into
  // 1 KiB blocks [row / 16][k / 64], the 64 16-byte chunks of a block in the order the lanes of the MFMA operand take
  // them ([(k % 64) / 16][row % 16]), so that a wave instruction fetches 1 KiB front to back.  Built on the device
  // when the handle is created (launch_block_weights).
  const int8_t *blocked;
};
// (An odd multiple of 256.  Without a selection: its result is no longer scalar to the compiler, and the K-block loop on row-major
// weights, whose descriptor has the stride in it, then went round a loop over the lanes' descriptors for each of its loads.)
__host__ __device__ inline int weight_row_stride(int k_pad) { return k_pad | 256; }

// Device memory through which the workgroups of a split GEMM (gemm_split.hip) hand over their sums: counters, which are zero
// between launches, and the sums.  Null: the GEMM is not split.  Launches on one stream follow one another and share it; so there
// is one for the null stream, and one for each stream of mi_stream_create, whose end the library sees, but not while that is
// captured: a replay may run beside the stream.
constexpr size_t kSplitCounterBytes = 1024, kSplitSumBytes = 256 * 256 * (4 * 64 + 16);  // 256 parts of 128 x 128 sums and row sums
constexpr size_t kSplitBytes = kSplitCounterBytes + kSplitSumBytes;
void *split_space(hipStream_t stream);
// For tests: the launches of split GEMMs of this thread so far, and the tile (as launch_gemm_split has it) and parts of the last.
struct SplitLaunches {
  int64_t count;
  int32_t tile, parts;
};
extern thread_local SplitLaunches t_split_launches;

// A: int8 activations [M][lda] (lda in bytes, multiple of 16, base 16-byte aligned, K % 16 == 0);
// W: packed weights (above); C: [M][ldc] elements, any n, ldc == n, any address of the element type.
int launch_gemm_requant(const int8_t *a, int64_t lda, int m, int k, const WeightView &w, int n,
                        const RequantParams &rq, int8_t *c, int64_t ldc, hipStream_t stream);
int launch_gemm_dequant(const int8_t *a, int64_t lda, int m, int k, const WeightView &w, int n,
                        const DequantParams &dq, float *c, int64_t ldc, hipStream_t stream);

// The same for activation rows of any length at any address, [m][k] without gaps, where that is quicker than a padded copy.
bool gemm_anyrow_takes(int m, int k, const WeightView &w, int n, const RequantParams &rq);
bool gemm_anyrow_takes(int m, int k, const WeightView &w, int n, const DequantParams &dq);
int launch_gemm_anyrow_requant(const int8_t *a, int m, int k, const WeightView &w, int n, const RequantParams &rq, int8_t *c,
                               hipStream_t stream);
int launch_gemm_anyrow_dequant(const int8_t *a, int m, int k, const WeightView &w, int n, const DequantParams &dq, float *c,
                               hipStream_t stream);

// Whether the launches above take m rows on the small tiles of gemm_short.hip, also where the decode kernels could: rows of any length and
// address by the last two, whole aligned chunks by the first two as well.
bool gemm_short_takes(int m, int k, const WeightView &w, int n, const RequantParams &rq);
bool gemm_short_takes(int m, int k, const WeightView &w, int n, const DequantParams &dq);

// Up to four weight matrices with the same K against the same activation rows as one launch; member i writes c[i] with row
// stride n[i].  gemm_group_tile: what the launch would run on, or null where the members are to be run one by one; lda: of the
// rows that it would be given; stream: theirs, since members are split on some only.
struct TileCost;
const TileCost *gemm_group_tile(int64_t lda, int m, int k, int count, const WeightView *w, const int *n, const RequantParams *rq,
                                hipStream_t stream);
const TileCost *gemm_group_tile(int64_t lda, int m, int k, int count, const WeightView *w, const int *n, const DequantParams *dq,
                                hipStream_t stream);
int launch_gemm_group_requant(const TileCost &tile, const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w,
                              const int *n, const RequantParams *rq, int8_t *const *c, hipStream_t stream);
int launch_gemm_group_dequant(const TileCost &tile, const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w,
                              const int *n, const DequantParams *dq, float *const *c, hipStream_t stream);

// Skinny-M path (m <= kGemvMaxRows): streams the weights once with 16-byte coalesced loads.
constexpr int kGemvMaxRows = 64;
constexpr int kGemvGroupMaxRows = 32;  // the group launches (several matrices, one launch) stop here
// 33..64 rows against at most 4096 channels come here where gemm_short.hip has no form for them (gemm_short_takes: up to 128 bytes of K, and the
// general rounding).  Of the others, this kernel's workgroups hold 16 channels each and the GEMM's smallest tile 64; against more
// channels the GEMM tiles have CUs enough and re-read the activations less.  us per launch at 64 rows, this path / 64 x 64 tiles and more: 4096 x 4096 8.8 / 11.0, 4096 x 11008 18.7 / 27.5, 768 x 3072 6.8 / 7.5, 6144 x 2048
// 9.2 / 7.6, 12288 x 4096 14.5 / 13.8; at 80 rows, where a form of the kernel with eight row groups existed: 4096 x 4096
// 11.9 / 9.8, 4096 x 11008 25.6 / 21.0, 768 x 3072 9.6 / 7.5.
constexpr int kGemvNarrowChannels = 4096;
inline bool gemv_takes_rows(int rows, int n) {
  return rows <= kGemvGroupMaxRows || (rows <= kGemvMaxRows && n <= kGemvNarrowChannels);
}
constexpr int kGemvDotRows = 2;  // up to here the v_dot4 kernel can run (it does for one row, and for two when the handle has no blocked copy), above it the MFMA kernel
int launch_gemv_requant(const int8_t *a, int64_t lda, int m, int k, const WeightView &w, int n,
                        const RequantParams &rq, int8_t *c, int64_t ldc, hipStream_t stream);

// Whether the two launches around here also take m rows of k bytes that are no whole 16-byte chunks, or not aligned to them,
// as they are; they then lie end to end (lda == k).
bool gemv_takes_any_rows(int m, int k, const WeightView &w, int n);

// 1..64 rows of the dynamic-quant MatMul (fp32 out) on the blocked weight copy (w.blocked must be there).
int launch_gemv_dequant(const int8_t *a, int64_t lda, int m, int k, const WeightView &w, int n,
                        const DequantParams &dq, float *c, int64_t ldc, hipStream_t stream);

// Up to four dynamic-quant MatMuls with the same K against the same activation rows, as one launch; member i writes
// c[i] (fp32) with row stride n[i].  For more than one row every member needs w.blocked.
int launch_gemv_group_dequant(const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w, const int *n,
                              const DequantParams *dq, float *const *c, hipStream_t stream);

// Up to four weight matrices with the same K against the same activation rows, as one launch (the grid is the
// concatenation of the members' grids); member i writes c[i] with row stride n[i].
int launch_gemv_group(const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w, const int *n,
                      const RequantParams *rq, int8_t *const *c, hipStream_t stream);

// Per-device set-up of the skinny-M kernels (function attributes); called by mi_init with the device current.
int gemv_prepare_device();

// Regroups packed row-major weights into the blocked copy described at WeightView::blocked.
int launch_block_weights(const int8_t *w, int n_pad, int k_pad, int ldw, int8_t *blocked, hipStream_t stream);

// Copies [rows][k] (row stride src_ld bytes) into a zero-padded [rows][k16] buffer, k16 = round_up(k, 16).
int launch_pad_rows(const int8_t *src, int64_t src_ld, int rows, int k, int8_t *dst, int k16, hipStream_t stream);

// im2col into [batch*out_h*out_w][k16] with K order (kh, kw, ic); out-of-image taps are `fill`, the K tail is zero.
int launch_im2col(const int8_t *in, const ConvGeom &g, int fill, int8_t *dst, int k16, hipStream_t stream);
// Dense convolution with kernel_h * kernel_w * in_c <= 64 and out_c <= 128, out_c % 4 == 0, straight from the image
// (no im2col buffer); w: packed row-major weights with row stride ldw, K order (kh, kw, ic).
int launch_conv_smallk(const int8_t *in, const ConvGeom &g, int fill, int k_true, const int8_t *w, int ldw,
                       const RequantParams &rq, int8_t *out, hipStream_t stream);
// Dense convolution on few input channels (in_c % 16 != 0, kernel_w * in_c <= 32, dilation_w 1), straight from the image
// with 16-byte loads; w: the weights as conv_rows_weights lays them out, in device memory.
constexpr int kConvRowsSteps = 8;  // at most this many 32-byte contraction steps
bool conv_rows_supported(const ConvGeom &g);
std::vector<int8_t> conv_rows_weights(const int8_t *w, int oc, int kernel_h, int kernel_w, int in_c);
int launch_conv_rows(const int8_t *in, const ConvGeom &g, int fill, const int8_t *w, const RequantParams &rq, int8_t *out,
                     hipStream_t stream);
// 1x1 convolution (stride 1, no padding) of a short contraction against few output channels, any alignment, pixels * k >= 16;
// w: the weights as conv_thin_weights lays them out, in device memory.
constexpr int64_t kConvThinMostPixels = 0x7fffffff - 65536;
bool conv_thin_supported(int k, int oc);
std::vector<int8_t> conv_thin_weights(const int8_t *w, int oc, int k);
int launch_conv_thin(const int8_t *in, int64_t pixels, int k, int oc, const int8_t *w, const RequantParams &rq, int8_t *out,
                     hipStream_t stream);
// Convolution of several taps on 16-channel-aligned images (in 16-byte aligned), its window's pixels in LDS, in the fast2 form
// without weight zero points; w: the weights as conv_window_weights lays them out, in device memory.  *taken false, and nothing
// launched, where the gathering GEMM is faster or the window does not fit.
bool conv_window_weights_wanted(const ConvGeom &g);
std::vector<int8_t> conv_window_weights(const ConvGeom &g, const int8_t *w);
int conv_window_prepare_device();  // called by mi_init with the device current
int launch_conv_window(const int8_t *in, const ConvGeom &g, const int8_t *fill16, const int8_t *w, const RequantParams &rq,
                       int8_t *out, hipStream_t stream, bool *taken);
// Depthwise conv + requantisation, weights pre-offset to int16 [KH*KW][C].  bias_folded = bias - zx8 * sum_t w16[t][c]
// (used by the channel-vectorised kernel, which reads out-of-image taps as zx8); rq.fast: the host proved the cheap
// rounding form exact for every channel.
int launch_conv_dw(const int8_t *in, const ConvGeom &g, const int16_t *w16, const int32_t *bias,
                   const int32_t *bias_folded, int zx8, const RequantParams &rq, int8_t *out, hipStream_t stream);
// The same with stride 1, a 3x3 or 5x5 window, int8 weights and out_c % 4 == 0 (in and out 4-byte aligned); w: the weights as
// conv_dw_rows_weights lays them out, par: {mult2, c2lo, c2hi, pre, shift}[out_c] of the one-multiply rounding form
// (RequantParams::fast2) with the bias of bias_folded.
bool conv_dw_rows_supported(const ConvGeom &g);
std::vector<int32_t> conv_dw_rows_weights(const int8_t *w, int ch, int ks);
int launch_conv_dw_rows(const int8_t *in, const ConvGeom &g, const int32_t *w, const int32_t *par, int zx8, int zo, int amin, int amax,
                        int8_t *out, hipStream_t stream);

// Host tensors of one call, in and out of device memory on the null stream (host_copy.hip).  `dev` holds a multiple of 16 bytes.
// The page-locked slots that the copies may go through (slot_pool.h) stay while a handle that has made such a call lives.
struct HostSlots;
class HostCopyUser {  // a member of every handle with such calls
 public:
  HostCopyUser() = default;
  HostCopyUser(const HostCopyUser &) = delete;
  HostCopyUser &operator=(const HostCopyUser &) = delete;
  ~HostCopyUser();

 private:
  friend class HostCopies;
  bool used_ = false;
};
class HostCopies {
 public:
  HostCopies(HostCopyUser *user, size_t most_bytes);  // most_bytes: of the largest tensor
  HostCopies(const HostCopies &) = delete;
  HostCopies &operator=(const HostCopies &) = delete;
  ~HostCopies();
  int in(void *dev, const void *host, size_t bytes);   // may return before the bytes are there; `host` is the caller's again
  int out(void *host, const void *dev, size_t bytes);  // returns when they are
 private:
  bool through_slots(const void *host, size_t bytes);
  HostCopyUser *user_;
  int size_;
  HostSlots *slots_ = nullptr;
};

// The requantising GEMM with its activation operand gathered from an NHWC image (in_c % 16 == 0): the im2col
// convolution without the buffer.  fill16: 16 bytes of the value out-of-image taps take, in device memory.
bool gemm_conv_supported(const ConvGeom &g, const void *in);
int launch_gemm_conv_requant(const int8_t *in, const ConvGeom &g, const int8_t *fill16, const WeightView &w,
                             const RequantParams &rq, int8_t *out, hipStream_t stream);

// DynamicQuant: per-block min/max partials, then quantise (every block re-reduces the partials).
constexpr int kDqMaxBlocks = 1024;
// slots: kDqSlotBytes of device memory, all zeros when made, through which the workgroups of the one-launch form meet.
constexpr int kDqFusedMost = 256;  // workgroups of the one-launch form: one per CU
// launch: the number of a launch among those on these slots, 1 .. kDqReplayed - 1 and never that of the launch before, or 0
// for a launch that may be replayed.
constexpr uint32_t kDqReplayed = 0x80000000u;
constexpr size_t kDqSlotBytes = sizeof(uint64_t) * (2 + 2 * kDqFusedMost);
// Page-locked host memory into which a run whose ticket is not 0 also writes {scale, zero point, min, max} as float /
// int32 bits in the low halves of kDqHostWords words, with the ticket in the high halves.
constexpr int kDqHostWords = 4;
struct DqHostNote {
  uint64_t *words;
  uint32_t ticket;
};
int launch_dynquant(const float *x, int64_t n, int symmetric, float2 *partials, void *slots, uint32_t launch,
                    const DqHostNote &note, mi_dq_params *params, int8_t *q, hipStream_t stream);
// One {scale, zero point} per contiguous run of `unit` elements; params has `segments` entries.
int launch_dynquant_segments(const float *x, int64_t segments, int64_t unit, int symmetric, mi_dq_params *params,
                             int8_t *q, hipStream_t stream);

}  // namespace mi
