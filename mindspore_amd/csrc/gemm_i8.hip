// int8 x int8 -> int32 GEMM on the gfx950 matrix cores (v_mfma_i32_32x32x32_i8) with fused epilogues:
//   EPI_REQUANT : + folded bias, - zw * input-row-sum, fixed-point requantise, + zo, clamp  -> int8
//                 (the arithmetic of MatmulInt8Opt / MatMulInt8_8x8_r, reference
//                  mindspore/ccsrc/plugin/device/cpu/kernel/nnacl/int8/matmul_int8.c:296-364)
//   EPI_DEQUANT : zero-point corrections, (sx*sw) * (float)acc, + bias, activation         -> fp32
//                 (DynamicMatmul4x16x4AIWI, .../nnacl/int8/dynamic_matmul_int8.c:99-143)
//
// Both operands are K-contiguous: activations A[M][K] and packed weights W[n_pad][k_pad].  A workgroup of four
// waves (2 x 2) owns a TILE_M x TILE_N output tile; the weight tile is the MFMA "A" operand (its rows are output
// channels) and the activation tile the "B" operand, so a lane ends up holding 4 consecutive output channels of
// one output row: the epilogue packs them into one 32-bit store, per-channel parameters are 16-byte loads, and
// the input-row sum a lane needs is the one it accumulated itself (v_dot4 against 0x01010101, or see RowSums).
//
// Several main loops, most of them moving tiles global -> LDS with asynchronous 16-byte-per-lane loads and reading operand
// fragments for the next K sub-step from LDS while the MFMAs of the current one run.  Handles hold their weights in
// 1 KiB matrix-core blocks beside the row-major form, and with those nearly every shape runs on K blocks of 128 bytes, on
// the tile that launch_pick_tile expects to be the quickest:
//   * gemm_kblock.hip: five LDS slots, one barrier per block; 256 x 256 and 192 x 256 tiles, one workgroup per CU, for the
//     large shapes, 128 x 128 tiles, two per CU, where fp32 stores have to overlap another tile's loop;
//   * gemm_ring.hip: a ring of stages that hold both operands, as deep as the LDS allows: every smaller tile;
//   * gemm_split.hip: the same with the K of a tile in parts, a workgroup each, where the tiles leave CUs idle;
//   * gemm_short.hip: 32 x 32 and 64 x 32 tiles whose K the waves share, where those fit the device about once;
//   * gemm_anyrow.hip: 64 x 64 tiles for activation rows that are no whole 16-byte chunks, where padding them first would cost
//     more than the product (gemm_short.hip takes such rows too);
//   * gemm_direct_body below, K steps of 64 bytes through NST LDS stages over row-major weights: short K, handles
//     without the blocked copy (whose large shapes run on gemm_kblock.hip's row-major form) and the convolution whose
//     activation operand is gathered from the image.
// Any K that is a multiple of 16: the weights are zero padded, so an activation chunk past K only has to be a valid
// read (it re-reads the row's last chunk).  LDS rows are XOR-swizzled in units of 16 bytes so that the 16-byte
// fragment reads of a wave are bank-conflict free.
#include <algorithm>

#include "gemm_core.h"

namespace mi {

template <int TN, int TM, bool HAS_ZW>
__device__ __forceinline__ void mma_frag(v16i (&acc)[TN][TM], int (&rowsum)[TM], const Frag<TN, TM> &f, int ones) {
  // ones: 0x01010101, or 0 when this lane's 16 activation bytes lie past K (they are then a re-read of valid
  // bytes, harmless for the products because the weights are zero there, but they must not enter the row sums)
  if (HAS_ZW) {
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      int t = rowsum[j];
      t = __builtin_amdgcn_sdot4(f.a[j].x, ones, t, false);
      t = __builtin_amdgcn_sdot4(f.a[j].y, ones, t, false);
      t = __builtin_amdgcn_sdot4(f.a[j].z, ones, t, false);
      t = __builtin_amdgcn_sdot4(f.a[j].w, ones, t, false);
      rowsum[j] = t;
    }
  }
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.w[i], f.a[j], acc[i][j], 0, 0, 0);
}

// Instruction-order hints for one K sub-step: spread the LDS operand reads between the MFMAs instead of issuing them
// in one burst, so that the matrix pipe always has the next MFMA queued.
template <int TN, int TM>
__device__ __forceinline__ void hint_interleave_reads() {
  // one read after each of the first MFMAs: the reads are all issued early in the sub-step, so their data has the
  // remaining MFMAs' time to arrive before the next sub-step needs it
  constexpr int kReads = TN + TM, kMfma = TN * TM;
  if constexpr (kMfma >= kReads) {
#pragma unroll
    for (int i = 0; i < kReads; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
    }
  } else {
#pragma unroll
    for (int i = 0; i < kMfma; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, kReads / kMfma, 0);
    }
  }
}

// =====================================================================================================================
// direct main loop: NST LDS stages x 64 bytes of K, asynchronous global -> LDS loads NST - 1 tiles ahead.
// NST = 4 in general (3 for short K, where a third workgroup per CU is worth more than depth); NST = 8 and 16 for handles
// without the blocked copy where few tiles walk a long K, a weight stream in which the number of bytes in flight per CU counts.
// OCC = workgroups the register allocation leaves room for on one CU (waves per SIMD).
// =====================================================================================================================
// CONV: the activation operand is not a matrix in memory but the im2col view of an NHWC image (in_c % 16 == 0): row m
// is output pixel m, and the 16-byte chunk at K offset k is 16 channels of tap k / in_c, fetched straight from the
// image, or from 16 bytes of the fill value when the tap lies outside the image (conv_int8.c:758-807,877).
template <typename Small>  // of strides, dilations and pads
struct ConvGatherOf {
  int in_h, in_w, in_c, out_w, out_hw;
  uint32_t magic_ic, magic_kw;  // ceil(2^32 / in_c), ceil(2^32 / kernel_w): exact quotients for dividends < 2^16
  Small stride_h, stride_w, dil_h, dil_w, pad_u, pad_l;
  int kernel_w;
};
typedef ConvGatherOf<int16_t> ConvGatherArgs;  // as it travels
typedef ConvGatherOf<int> ConvGather;
__device__ __forceinline__ ConvGather open(const ConvGatherArgs &c) {
  ConvGather cv{c.in_h, c.in_w, c.in_c, c.out_w, c.out_hw, c.magic_ic, c.magic_kw, c.stride_h, c.stride_w, c.dil_h, c.dil_w,
                c.pad_u, c.pad_l, c.kernel_w};
  // (in registers for good: left to itself the compiler takes the main loop's out of their shared word in every K step.  us at long K:
  // 1 x 27 x 27, 256 -> 256, 5x5 at stride 2 21.2 -> 20.8, with left shifts 22.2 -> 21.4; 16 x 14 x 14, 256 -> 512, 3x3 at stride 2, with
  // left shifts 10.25 -> 10.0)
  asm volatile("" : "+s"(cv.dil_h), "+s"(cv.dil_w));
  return cv;
}
// As GemmCall, of a convolution whose output pixels are the rows.
struct ConvCall {
  const int8_t *in, *w, *fill16;
  int8_t *c;
  int m, n, k;
  ConvGatherArgs cv;
  RequantCall epi;
};
static_assert(sizeof(ConvCall) <= kShortArgs, "see launch_args.h");

template <int TILE_N, int TILE_M, int EPI, bool HAS_ZW, bool FAST, int NST, bool CONV>
__device__ __forceinline__ void gemm_direct_body(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                                                 const ConvGather &cv, const int8_t *fill16) {
  constexpr int BKD = 64, PD = NST - 1;  // PD: prefetch distance in K steps
  static_assert(NST >= 3, "the loop keeps NST - 1 >= 2 tiles in flight");
  auto wrap = [](int x) { return x >= NST ? x - NST : x; };  // stage index after an increment of at most NST
  constexpr int WN = TILE_N / 2, WM = TILE_M / 2, TN = WN / 32, TM = WM / 32;
  constexpr int STAGE = (TILE_N + TILE_M) * BKD;
  constexpr int WPW = TILE_N / 16 / 4, APW = TILE_M / 16 / 4, LPW = WPW + APW;  // 1 KiB blocks per wave and tile
  static_assert(WPW >= 1 && APW >= 1, "tile too small");
  static_assert(EPI != EPI_REQUANT || TN != 2 || TM != 2 || NST * STAGE >= kEpiArrays * TILE_N * 4 + 16384,
                "the workgroup's output staging tile must fit the main loop's LDS");
  static_assert(EPI == EPI_REQUANT ? (TN != 4 || TM != 4 || NST * STAGE >= kEpiArrays * TILE_N * 4 + 4 * 16384)
                                   : NST * STAGE >= kEpiArrays * TILE_N * 4 + 4 * epi_stage_bytes<EPI, TM>(),
                "the epilogue staging must fit the main loop's LDS");
  __shared__ __attribute__((aligned(1024))) char lds[NST * STAGE];

  int tile_m, tile_n;
  tile_coords<!CONV>(g, &tile_m, &tile_n);
  const int m0 = tile_m * TILE_M, n0 = tile_n * TILE_N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int r = lane & 31, h = lane >> 5;
  const int ktiles = (g.k + BKD - 1) / BKD;  // the zero padding of the weights past K needs no MFMAs
  const int kchunks = g.k >> 4;
  EpiParams<TILE_N, EPI, FAST> epi;
  epi.fetch(rq, dq, n0, g.n, tid);
  DeqInput<TM> din;
  if (EPI == EPI_DEQUANT) din.fetch_rows(dq, m0 + wm * WM, r, g.m);

  // loader: a 1 KiB block holds 16 rows x 64 B.  Lane L fills slot (L & 3) of row (L >> 2) of its block, i.e. it
  // fetches logical chunk (L & 3) ^ swizzle(row), swizzle(row) = (row >> 1) & 3.
  const int drow = lane >> 2;
  const int dchunk = (lane & 3) ^ ((lane >> 3) & 3);
  const int8_t *wsrc = g.w + (int64_t)(n0 + wave * WPW * 16 + drow) * g.ldw + dchunk * 16;
  const int8_t *asrc[APW];
  int ih0[CONV ? APW : 1], iw0[CONV ? APW : 1];
#pragma unroll
  for (int i = 0; i < APW; ++i) {
    int m = m0 + (wave * APW + i) * 16 + drow;
    m = m < g.m ? m : g.m - 1;
    if (CONV) {
      const int b = m / cv.out_hw, rem = m - b * cv.out_hw;
      const int oh = rem / cv.out_w, ow = rem - oh * cv.out_w;
      ih0[i] = oh * cv.stride_h - cv.pad_u;
      iw0[i] = ow * cv.stride_w - cv.pad_l;
      // address of (ih0, iw0, channel 0); only dereferenced for taps inside the image
      asrc[i] = g.a + (((int64_t)b * cv.in_h + ih0[i]) * cv.in_w + iw0[i]) * cv.in_c;
    } else {
      asrc[i] = g.a + (int64_t)m * g.lda;
    }
  }
  // A has exactly K valid bytes per row (the weights are zero padded, A is the caller's): a 16-byte chunk past K is
  // fetched from the row's last chunk instead
  const int a_last = (kchunks - 1) * 16;
  auto dma_tile = [&](int stage, int kt) {
    char *sw = lds + stage * STAGE + wave * WPW * 1024;
    char *sa = lds + stage * STAGE + TILE_N * BKD + wave * APW * 1024;
#pragma unroll
    for (int i = 0; i < WPW; ++i) async_copy16(wsrc + (int64_t)i * 16 * g.ldw + kt * BKD, sw + i * 1024);
    int koff = kt * BKD + dchunk * 16;
    if (CONV) {
      const uint32_t tap = __umulhi((uint32_t)koff, cv.magic_ic);
      const int ic = koff - (int)tap * cv.in_c;
      const uint32_t kh = cv.kernel_w == 1 ? tap : __umulhi(tap, cv.magic_kw);
      const int dh = (int)kh * cv.dil_h, dw = ((int)tap - (int)kh * cv.kernel_w) * cv.dil_w;
      const int tap_off = (dh * cv.in_w + dw) * cv.in_c + ic;
      const bool in_k = koff < g.k;  // past K the weights are zero: any 16 readable bytes will do
#pragma unroll
      for (int i = 0; i < APW; ++i) {
        const int ih = ih0[i] + dh, iw = iw0[i] + dw;
        const bool inside = in_k && (unsigned)ih < (unsigned)cv.in_h && (unsigned)iw < (unsigned)cv.in_w;
        async_copy16(inside ? asrc[i] + tap_off : fill16, sa + i * 1024);
      }
      return;
    }
    koff = koff < a_last ? koff : a_last;
#pragma unroll
    for (int i = 0; i < APW; ++i) async_copy16(asrc[i] + koff, sa + i * 1024);
  };

  v16i acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = (int)kAccBias;  // see kAccBias
  int rowsum[TM];
#pragma unroll
  for (int j = 0; j < TM; ++j) rowsum[j] = 0;

  // operand fragments: this lane's rows are r + multiples of 32, so its swizzle is a lane constant
  const int frag_swz = (r >> 1) & 3;
  const int w_off = (wn * WN + r) * BKD, a_off = TILE_N * BKD + (wm * WM + r) * BKD;
  Frag<TN, TM> f0, f1;
  auto read_frag = [&](Frag<TN, TM> &f, int stage, int s) {
    const char *base = lds + stage * STAGE + (((2 * s + h) ^ frag_swz) << 4);
#pragma unroll
    for (int i = 0; i < TN; ++i) f.w[i] = *reinterpret_cast<const v4i *>(base + w_off + i * 32 * BKD);
#pragma unroll
    for (int j = 0; j < TM; ++j) f.a[j] = *reinterpret_cast<const v4i *>(base + a_off + j * 32 * BKD);
  };
  // One 64-byte K step on LDS stage `st` (tile kt).  On entry f0 holds sub-step 0 of this stage.
  //   sub-step 0 : MFMAs on f0 while f1 <- sub-step 1 of this stage
  //   barrier    : first wait until at most (PD - 2) * LPW of this wave's loads are outstanding (loads complete in
  //                order, so that is "tile kt+1 has landed, later tiles may still be in flight"), then meet the other
  //                waves: now tile kt+1 is complete in LDS and nobody reads stage st-1 (tile kt-1) any more
  //   sub-step 1 : refill that stage with tile kt+PD, f0 <- sub-step 0 of tile kt+1, MFMAs on f1
  // With more than four stages the loads past the end of K re-fetch the last tile into a stage nobody reads again,
  // which keeps the outstanding-load count the same in every step; with up to four the last steps are separate
  // bodies without loads (see below).
  auto step = [&](int kt, int st) {
    read_frag(f1, st, 1);
    mma_frag<TN, TM, HAS_ZW>(acc, rowsum, f0, (kt * 4 + h < kchunks) ? 0x01010101 : 0);
    hint_interleave_reads<TN, TM>();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((PD - 2) * LPW) : "memory");
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const int nxt = kt + PD < ktiles ? kt + PD : ktiles - 1;
    read_frag(f0, wrap(st + 1), 0);
    dma_tile(wrap(st + PD), nxt);
    mma_frag<TN, TM, HAS_ZW>(acc, rowsum, f1, (kt * 4 + 2 + h < kchunks) ? 0x01010101 : 0);
    {
      // operand reads first (the next sub-step waits for them), the loads of tile kt+3 behind them (they have
      // almost three steps to land)
      constexpr int kMfma = TN * TM, kReads = TN + TM;
      if constexpr (kMfma >= kReads + LPW) {
#pragma unroll
        for (int i = 0; i < kReads; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
        }
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // global -> LDS load issue
        }
      } else {
#pragma unroll
        for (int i = 0; i < kMfma; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, (kReads + kMfma - 1) / kMfma, 0);
          __builtin_amdgcn_sched_group_barrier(0x020, (LPW + kMfma - 1) / kMfma, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int t = 0; t < PD; ++t) dma_tile(t, t < ktiles ? t : ktiles - 1);
  if (EPI == EPI_DEQUANT) din.fetch_tensor(dq);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((PD - 1) * LPW) : "memory");
  read_frag(f0, 0, 0);
  if constexpr (NST <= 4) {
    // The last PD steps have bodies of their own that load nothing: with a dozen K steps, as in the K = 768 shapes,
    // re-fetching the last tile PD times is a fifth of the operand traffic.  REM = tiles after this one; the tiles
    // still in flight at its wait are kt+2 .. the last one.
    auto tail_step = [&](int kt, int st, auto rem_c) {
      constexpr int REM = decltype(rem_c)::value;
      read_frag(f1, st, 1);
      mma_frag<TN, TM, HAS_ZW>(acc, rowsum, f0, (kt * 4 + h < kchunks) ? 0x01010101 : 0);
      hint_interleave_reads<TN, TM>();
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (REM >= 1) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((REM - 1) * LPW) : "memory");
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        read_frag(f0, wrap(st + 1), 0);
      }
      mma_frag<TN, TM, HAS_ZW>(acc, rowsum, f1, (kt * 4 + 2 + h < kchunks) ? 0x01010101 : 0);
      hint_interleave_reads<TN, TM>();
      __builtin_amdgcn_sched_barrier(0);
    };
    int kt = 0, st = 0;
    for (; kt + PD < ktiles; ++kt, st = wrap(st + 1)) step(kt, st);
    if constexpr (PD >= 3) {
      if (ktiles - 1 - kt == 2) {
        tail_step(kt, st, std::integral_constant<int, 2>());
        ++kt;
        st = wrap(st + 1);
      }
    }
    if (ktiles - 1 - kt == 1) {
      tail_step(kt, st, std::integral_constant<int, 1>());
      ++kt;
      st = wrap(st + 1);
    }
    tail_step(kt, st, std::integral_constant<int, 0>());
  } else {
    for (int kt = 0, st = 0; kt < ktiles; ++kt, st = wrap(st + 1)) step(kt, st);
  }
  // (also: every load must have landed before the LDS is reused below or handed to another workgroup)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  epi.to_lds(reinterpret_cast<int *>(lds), tid);
  gemm_epilogue<TILE_N, TN, TM, EPI, HAS_ZW, FAST, kAccBias>(
      acc, rowsum, g, rq, dq, din, reinterpret_cast<const int *>(lds),
      lds + kEpiArrays * TILE_N * 4 + wave * epi_stage_bytes<EPI, TM>(), lds + kEpiArrays * TILE_N * 4, n0, m0,
      n0 + wn * WN, m0 + wm * WM, r, h);
}

template <int TILE_N, int TILE_M, int EPI, bool HAS_ZW, bool FAST, int NST, int OCC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void gemm_direct_kernel(GemmCall<EPI> call) {
  GemmArgs g;
  RequantParams rq;
  DequantParams dq;
  call.open(&g, &rq, &dq);
  gemm_direct_body<TILE_N, TILE_M, EPI, HAS_ZW, FAST, NST, false>(g, rq, dq, ConvGather{}, nullptr);
}

// The same GEMM with the activation operand gathered from an NHWC image (no im2col buffer).
template <int TILE_N, int TILE_M, bool HAS_ZW, bool FAST, int NST, int OCC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void gemm_conv_kernel(ConvCall call) {
  call.epi.load_now();
  asm volatile("" ::"s"(call.in), "s"(call.w), "s"(call.fill16), "s"(call.c), "s"(call.m), "s"(call.n), "s"(call.k), "s"(call.cv.in_h), "s"(call.cv.in_w),
               "s"(call.cv.in_c), "s"(call.cv.out_w), "s"(call.cv.out_hw), "s"(call.cv.magic_ic), "s"(call.cv.magic_kw), "s"(call.cv.kernel_w));
  const int k_pad = padded_k(call.k);
  const GemmArgs g{call.in, 0, call.m, call.k, call.w, weight_row_stride(k_pad), k_pad, nullptr, call.n,
                   (call.m + TILE_M - 1) / TILE_M, (call.n + TILE_N - 1) / TILE_N, call.c, call.n, 0, 0};
  gemm_direct_body<TILE_N, TILE_M, EPI_REQUANT, HAS_ZW, FAST, NST, true>(g, call.epi.open(call.n), DequantParams{}, open(call.cv),
                                                                         call.fill16);
}

// ---- host side -----------------------------------------------------------------------------------------------
template <int TILE_N, int TILE_M, int EPI, bool HAS_ZW, bool FAST, int NST = 4, int OCC = 1>
static int launch_cfg(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  const auto call = GemmCall<EPI>::of(g, g.w, TILE_N, TILE_M, rq, dq);
  auto kern = gemm_direct_kernel<TILE_N, TILE_M, EPI, HAS_ZW, FAST, NST, OCC>;
  launch_kernel(kern, call.grid(), dim3(256), 0, stream, call);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

// The K-block loops on the blocked weight copy, by what a launch is expected to take: rounds x (a + b x K blocks of 128
// bytes), a round being as many tiles as the device runs at once.  A tile lasts longer the larger it is, but less than in
// proportion to its area -- small tiles are bound by the way from the L2 into LDS, about 110 GB/s a CU -- so the smallest
// tile that fits the device in one round wins, and beyond one round the one that wastes least of its last.  a and b
// (us) are fitted to launches with weights streamed from HBM at 6 and 32 K blocks.
struct TileCost {
  bool ring;
  int tn, tm, per_round;
  float a, b;
};
constexpr TileCost kTileCosts[] = {
    {true, 1, 1, 256, 2.8f, 0.25f},  {true, 1, 2, 256, 2.9f, 0.36f},  {true, 2, 2, 256, 3.0f, 0.57f},
    {true, 3, 2, 256, 3.2f, 0.84f},  {true, 2, 4, 256, 3.5f, 0.95f},  {true, 4, 2, 256, 3.6f, 0.96f},
    {false, 2, 2, 512, 5.0f, 1.02f}, {false, 3, 4, 256, 5.0f, 1.22f}, {false, 4, 4, 256, 5.0f, 1.55f},
};
// For `count` matrices of n[i] channels whose tiles share a launch.
static const TileCost &cheapest_tile(int m, int k, int count, const int *n, float *least) {
  const TileCost *best = nullptr;
  const int kblocks = (k + 127) / 128;
  for (const TileCost &t : kTileCosts) {
    int64_t columns = 0;
    for (int i = 0; i < count; ++i) columns += (n[i] + 64 * t.tn - 1) / (64 * t.tn);
    const int64_t tiles = (int64_t)((m + 64 * t.tm - 1) / (64 * t.tm)) * columns;
    const float cost = (float)((tiles + t.per_round - 1) / t.per_round) * (t.a + t.b * (float)kblocks);
    if (best == nullptr || cost < *least) best = &t, *least = cost;
  }
  return *best;
}
// K split over the workgroups of a tile (gemm_split.hip): expected to take a + b x K blocks of a part + 1.7 us for the sums' way
// through memory + `part` for every part after the first + `wg` for every workgroup, whose sums all go that way at once.  b_far:
// where the weights are too large to be in the caches, which holds up unsplit launches too, but not 64 x 64 tiles of more rows than
// the weights stream past (kStreamRowTiles); b_two, where it is not 0: with two row tiles.  The margins are for what a and b do not
// know.  us per launch, unsplit / split, weights from memory: 65 x 3328 x 8368 24.8 / 16.6, 128 x 4096 x 11008 26.3 / 18.3,
// 128 x 4096 x 4096 10.7 / 9.8, 64 x 6000 x 8000 21.9 / 15.8, 100 x 1024 x 4096 9.5 / 7.8, 138 x 1408 x 5632 10.9 / 9.3,
// 300 x 1024 x 8192 14.4 / 10.5, 1000 x 512 x 8192 14.9 / 12.2, 512 x 4096 x 11008 38.1 / 35.7, 176 x 2407 x 7360 18.75 / 13.6; not
// taken: 200 x 1024 x 2048 5.8 / 7.0, 197 x 768 x 3072 7.43 / 7.46, 161 x 1280 x 3120 7.86 / 7.87, 512 x 4096 x 4096 13.3 / 18.5,
// 256 x 4096 x 4096 10.0 / 13.2, 800 x 1280 x 5120 14.5 / 15.6, and for b_two 144 x 3756 x 10336 20.7 / 31.2, 199 x 2252 x 7888 15.5 /
// 19.1, 232 x 2905 x 10016 24.05 / 28.1.
struct SplitCost {
  int tn, tm, most_parts;
  float a, b, b_far, b_two, part, wg;
};
constexpr SplitCost kSplitCosts[] = {{1, 1, 8, 2.8f, 0.25f, 0.285f, 0, 0.25f, 0.008f},
                                     {1, 2, 8, 2.9f, 0.36f, 0.41f, 0.55f, 0.35f, 0.016f},
                                     {2, 2, 2, 3.0f, 0.57f, 0.57f, 0, 0.5f, 0.022f}};
constexpr int64_t kFarWeights = 16 << 20;
// The tile, the number of parts and what they are expected to take, or null where the unsplit launch on `whole` is expected to be as quick.
static const SplitCost *choose_split(int m, int k, int n, const TileCost &whole, float cost, int *parts, float *split_cost) {
  const SplitCost *best = nullptr;
  const int kblocks = (k + 127) / 128;
  const bool far = (int64_t)n * k >= kFarWeights;
  for (const SplitCost &t : kSplitCosts)
    if (far && whole.ring && whole.tn == t.tn && whole.tm == t.tm && (t.tm > 1 || (m + 63) / 64 <= kStreamRowTiles))
      cost *= (t.a + t.b_far * (float)kblocks) / (t.a + t.b * (float)kblocks);
  float least = (far ? 0.99f : 0.9f) * cost;
  for (const SplitCost &t : kSplitCosts) {
    const int64_t rows = (m + 64 * t.tm - 1) / (64 * t.tm), tiles = rows * ((n + 64 * t.tn - 1) / (64 * t.tn));
    const int most = (int)std::min<int64_t>(256 / tiles, std::min(kblocks, t.most_parts));
    const float b = rows == 2 && t.b_two > 0 ? t.b_two : far ? t.b_far : t.b;
    for (int p = 2; p <= most; ++p) {
      const float c = t.a + b * (float)((kblocks + p - 1) / p) + 1.7f + t.part * (float)(p - 1) + t.wg * (float)(tiles * p);
      if (c < least) best = &t, least = c, *parts = p;
    }
  }
  if (best != nullptr) *split_cost = least;
  return best;
}
// The tile of gemm_short.hip that is quicker than what else there is, or 0; and what it is expected to take (us, fitted like kTileCosts to 756 shapes
// with weights from memory, median error 3 to 5 %).
// One 32 x 32 tile a CU, of four waves up to 12 K blocks and of eight beyond, or, from 7 blocks on, one of 64 channels x 32 rows: the
// second workgroup of a CU competes for the operands' way into it, about 100 GB/s.  With fewer blocks the launch is most of the time, and
// several tiles a CU still pay, with fp32 output, whose stores they spread, more of them.  us per launch, the quickest otherwise / this:
// 33 x 1024 x 4096 7.05 / 5.2, 65 x 3072 x 1024 (288 tiles of 32 x 32, 144 of 64 x 32) 4.65 / 4.20, 128 x 4096 x 4096 (256 of 64 x 32) 9.9 / 8.9,
// 1000 x 500 x 256 3.69 / 3.45 (512), 700 x 1024 x 512 (fp32) 4.8 / 4.24 (704); not taken: 160 x 3072 x 768 4.20 / 4.34 (480), 333 x 1536 x 512
// 3.97 / 4.06 (528), 512 x 768 x 128 3.17 / 3.38, 200 x 3072 x 1024 4.47 / 5.24 (336 of 64 x 32: 6.7), 200 x 4096 x 4096 10.1 / 14.6 (448 of 64 x 32),
// 65 x 4096 x 11008 18.5 / 18.8.
struct ShortTile {
  int tile;  // as launch_gemm_short has it
  float cost;
};
// The most K blocks of up to 32 rows, which the decode kernels read K in 16 channels a workgroup for, three times 16 from 8192 channels on:
// quick at long K, and quicker the fewer the rows, as long as one round of their workgroups holds all channels.  Time of this relative to
// theirs, weights from memory, over rows of any length and int8 and fp32 output:
//   up to 4 rows   768 channels 4 blocks 0.91 - 1.01, 6 0.95 - 1.08, 10 1.23 - 1.29; 4096 3 0.91 - 1.02, 5 1.04 - 1.15, 12 1.16 - 1.39;
//                  6144 7 0.9 - 1.0, 9 1.05 - 1.09; 12288 3 0.96 - 1.03, 5 1.05; 16384 6 0.83 - 0.85
//   up to 8        768 6 0.92 - 0.98, 9 1.01 - 1.12; 2048 6 0.89 - 1.06, 9 1.12 - 1.27; 4096 5 0.99 - 1.04, 9 1.16 - 1.22; 6144 12 0.92 - 1.05;
//                  8192 5 0.94 - 0.99, 8 1.02 - 1.09; 24576 6 0.9
//   up to 32       512 12 0.82 - 0.97; 768 12 0.91 - 1.06; 2048 8 0.83 - 0.99, 10 0.96 - 1.10; 4096 8 0.86 - 0.98, 10 0.93 - 1.09; 6144 12 0.68 -
//                  0.99; 8192 8 0.71 - 1.01; 17 rows and more 8192 12 0.86 - 0.92
// us: 4 x 768 x 1277 3.51 / 4.41, 8 x 2048 x 1520 3.66 / 4.48, 4 x 768 x 448 3.27 / 2.98, 16 x 5000 x 768 4.95 / 3.41, 32 x 24000 x 768 10.1 / 6.1.
static int few_rows_most_blocks(int m, int n) {
  const bool second_round = (n > kGemvNarrowChannels && n < 8192) || n > 12288;
  if (m <= 4) return n <= 2048 ? 4 : second_round ? 7 : 3;
  if (m <= 8) return n <= 2048 ? 6 : second_round ? 12 : 5;
  return n <= 768 || second_round || (m > 16 && n >= 8192) ? 12 : 8;
}
static ShortTile short_tile(int m, int k, int n, bool requant) {
  const int kb = (k + 127) / 128;
  const int64_t rows = (m + 31) / 32, small = rows * ((n + 31) / 32), wide = rows * ((n + 63) / 64);
  if (kb < 2 || m <= kGemvDotRows) return {0, 0};
  const auto cost = [kb](int64_t tiles, float a, float k, float block, float tile) {
    return a + k * (float)kb + (float)tiles / 256.0f * (block * (float)kb + tile);
  };
  const auto four = [&] { return ShortTile{41, cost(small, 2.68f, 0.083f, 0.094f, 0.22f)}; };
  if (m <= kGemvGroupMaxRows)  // (tiles: 16 x 8192 x 1536, 256 of them, 4.72 / 4.92; 16 x 12288 x 1024, 384, 4.52 / 5.16)
    return kb <= few_rows_most_blocks(m, n) && small <= (kb <= 6 ? 768 : kb <= 8 || m > 16 ? 256 : 224) ? four() : ShortTile{0, 0};
  if (small <= 256) return kb <= 12 ? four() : ShortTile{81, cost(small, 2.53f, 0.08f, 0.04f, 0.47f)};
  if (kb < 7) return small <= (!requant ? 768 : kb == 2 ? 256 : kb < 6 ? 512 : 448) ? four() : ShortTile{0, 0};
  return wide <= 256 && kb <= 64 ? ShortTile{82, cost(wide, 3.6f, 0.089f, 0.1f, -0.28f)} : ShortTile{0, 0};
}
// The same for rows in whole chunks, where nothing is copied for the other tiles: five row tiles of int8 that nearly fill the device read the
// weights five times to three, up to 20 K blocks.  Time of this relative to theirs: 160 x 3072 x 1280 1.10 (5.71 / 5.15 us), 160 x 3200 x 2560
// 1.09, 160 x 2880 x 2560 1.07, 129 x 3200 x 2560 1.06; not so 160 x 2500 x 2048 0.98, 160 x 2881 x 3072 0.94, 160 x 3200 x 3072 1.04, with fp32
// output 160 x 3072 x 1280 1.01, 192 x 2560 1.0, 128 x 4096 0.9; rows that would have to be copied 0.76 - 0.9.
static ShortTile short_tile_of_chunks(int m, int k, int n, bool requant) {
  const bool full = requant && (m + 31) / 32 == 5 && (n + 63) / 64 * 5 > 224 && k <= 20 * 128;
  const ShortTile t = short_tile(m, k, n, requant);
  return full && t.tile == 82 ? ShortTile{0, 0} : t;
}
// From K = 4096 on, more rows than the decode kernels take stay with K in parts (gemm_split.hip) on the streams that have memory for
// that: its tests hold it to them.  128 x 1024 x 4096 7.7 us in parts, 5.3 here.
static bool short_goes_first(int m, int k) { return m <= kGemvMaxRows || k < 4096; }

// (the K-block loaders address activation rows with 32-bit offsets from the tile's first row)
static bool kblock_takes(int k, int64_t lda) { return k >= 128 && lda < (1 << 23); }

template <int EPI, bool HAS_ZW, bool FAST>
static int launch_pick_tile(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                            hipStream_t stream) {
  const int64_t tiles_l = (int64_t)((g.m + 255) / 256) * ((g.n + 255) / 256);
  const int64_t tiles_m = (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128);
  const bool kblock_ok = kblock_takes(g.k, g.lda);
  // With a blocked weight copy: any long K, and short ones as long as 128 x 128 tiles are enough for one round.  us per
  // launch, weights from HBM, before -> now: 512 x 12288 x 4096 37.0 -> 30.1, 512 x 4096 x 4096 19.4 -> 14.5,
  // 512 x 4096 x 11008 48.4 -> 36.9, 2048 x 12288 x 4096 (fp32) 110.9 -> 99.2, 2048 x 4096 x 11008 (fp32) 92 -> 81.6,
  // 256 x 4096 x 4096 14.0 -> 10.9, 100 x 12288 x 4096 20.0 -> 15.8, 197 x 768 x 3072 (fp32) 9.3 -> 7.6,
  // 4096 x 768 x 3072 (fp32) 16.7 -> 14.7, 128 x 768 x 768 5.1 -> 4.3.
  // With fp32 output and a short K two workgroups per CU overlap one's stores with the other's loop: 4096 x 768 x 768 7.6
  // against 7.9 us.
  if (g.wb != nullptr && kblock_ok && (g.k >= 1024 || tiles_m <= 256)) {
    const bool short_form = EPI == EPI_REQUANT ? FAST : !FAST;
    const int in_short = short_form ? short_tile_of_chunks(g.m, g.k, g.n, EPI == EPI_REQUANT).tile : 0;
    if (in_short != 0 && short_goes_first(g.m, g.k)) return launch_gemm_short(in_short, false, EPI == EPI_REQUANT, HAS_ZW, g, rq, dq, stream);
    if (EPI == EPI_DEQUANT && g.k < 1024 && tiles_m >= 128) return launch_gemm_kblock(22, false, HAS_ZW, FAST, g, rq, dq, stream);
    float cost;
    const TileCost &t = cheapest_tile(g.m, g.k, 1, &g.n, &cost);
    if (EPI == EPI_REQUANT ? FAST : !HAS_ZW) {  // (the forms that gemm_split.hip has)
      int parts;
      const SplitCost *split = choose_split(g.m, g.k, g.n, t, cost, &parts, &cost);
      void *space = split != nullptr ? split_space(stream) : nullptr;
      if (space != nullptr)
        return launch_gemm_split(10 * split->tn + split->tm, parts, EPI == EPI_REQUANT, HAS_ZW, FAST, g, rq, dq, space, stream);
    }
    if (in_short != 0) return launch_gemm_short(in_short, false, EPI == EPI_REQUANT, HAS_ZW, g, rq, dq, stream);
    return t.ring ? launch_gemm_ring(10 * t.tn + t.tm, EPI == EPI_REQUANT, HAS_ZW, FAST, g, rq, dq, stream)
                  : launch_gemm_kblock(10 * t.tn + t.tm, EPI == EPI_REQUANT, HAS_ZW, FAST, g, rq, dq, stream);
  }
  // From here on mostly handles without the blocked copy.
  // a few activation rows against a big weight matrix: one row of 64 x 64 tiles, deep prefetch (HBM-bound)
  if (g.m <= 64 && g.k_pad >= 1024) return launch_cfg<64, 64, EPI, HAS_ZW, FAST, 16>(g, rq, dq, stream);
  if (g.m <= 128 && g.k_pad >= 1024) return launch_cfg<64, 128, EPI, HAS_ZW, FAST, 8>(g, rq, dq, stream);
  // Few tiles and a long K: every workgroup walks its whole K alone at the pace of its own loop (a 64 x 64 tile takes
  // about 0.2 us per 64 bytes of K, a 64 x 128 tile 0.3, a 128 x 128 tile 0.6 per 128 bytes, whatever the number of
  // workgroups up to one per CU), so the smallest tile that still fits the device in one round wins, on eight stages
  // (three steps in flight leave a lone workgroup waiting on memory).  Measured with the weights streamed from HBM
  // (us per launch): 256 x 4096 x 4096 23.2 -> 15.6, 256 x 4096 x 11008 55.0 -> 35.7, 384 x 4096 x 4096 42.8 -> 19.5,
  // 512 x 4096 x 4096 22.2 -> 19.3, 512 x 3072 x 4096 41.2 -> 19.1, 2048 x 768 x 3072 31.8 -> 14.0,
  // 256 x 8192 x 2048 13.6 -> 12.5; with the weights in the L2s 300 x 4096 x 2048 16.4 -> 11.0,
  // 640 x 2048 x 1024 8.5 -> 6.9, and 5 % slower where fewer than a hundred tiles find them there
  // (512 x 768 x 3072: 8.5 -> 9.0).  Sixteen stages are no better than eight.
  if (g.k_pad >= 1024) {
    const int64_t cols64 = (g.n + 63) / 64;
    if ((int64_t)((g.m + 63) / 64) * cols64 <= 256) return launch_cfg<64, 64, EPI, HAS_ZW, FAST, 8, 2>(g, rq, dq, stream);
    // (against the 128 x 128 K-block tiles at K = 1024 the 64 x 128 tile is 15 % ahead on streamed weights and 4-9 %
    //  behind on cache-resident ones -- 512 x 4096 x 1024: 7.1 -> 7.7 us -- so it starts at K = 2048, where it is
    //  10-13 % ahead on those too: 512 x 4096 x 4096 20.4 -> 17.8 us, 2048 x 768 x 3072 13.9 -> 12.3 us)
    if (g.k_pad >= 2048 && (int64_t)((g.m + 127) / 128) * cols64 <= 256)
      return launch_cfg<64, 128, EPI, HAS_ZW, FAST, 8>(g, rq, dq, stream);
  }
  // The 256 x 256 tile does a unit of work in little more than half the time the 128 x 128 tiles need, so with int8
  // output it is taken as soon as the 128 x 128 tiles would no longer fit the device in one go (more than 512 of
  // them, i.e. more than 128 large tiles): 2304 x 4096 x 4096 51.6 -> 41.2 us, 2816 x 4096 x 1024 20.4 -> 17.8 us;
  // at exactly 128 large tiles the 512 small ones win (2048 x 4096 x 4096: 35.5 against 39.8 us).
  // The fp32 epilogue writes four times the bytes: below one 256 x 256 tile per CU it is worth more to overlap it
  // with another workgroup's main loop than to save operand traffic.
  if (tiles_l >= (EPI == EPI_DEQUANT ? 256 : 129) && kblock_ok)
    return launch_gemm_kblock(44, EPI == EPI_REQUANT, HAS_ZW, FAST, g, rq, dq, stream);
  // From one 128 x 128 tile per two CUs on: the K-block loop on 128 x 128 tiles, two workgroups per CU.  Whole
  // cache lines per load and one barrier per 128 bytes of K make its main loop about a third shorter than the
  // 64-byte-step loop below; two workgroups per CU instead of three make a round of tiles more expensive.  Measured on
  // 21 int8-output shapes from 768 x 3072 x 768 to 1536 x 1536 x 6144: 0-25 % faster (2048^3 15.3 -> 13.8 us,
  // 512 x 8192 x 1024 13.8 -> 10.5 us), 2 % slower only at K = 32.  With fp32 output the epilogue weighs more: it wins
  // where the loop dominates (K >= 2048: 4096 x 768 x 3072 21.0 -> 19.0 us) and where the three-per-CU form below
  // has all its tiles store in the same moment (>= 768 tiles: 4096 x 3072 x 768 25.9 -> 24.4 us), and with at most
  // one tile per CU (4096 x 768 x 768: 8.6 -> 8.3 us); it loses on 576 tiles at K = 768 (18.4 against 22.2 us).
  if (tiles_m >= 128 && kblock_ok &&
      (EPI == EPI_REQUANT || g.k >= 2048 || tiles_m >= 768 || tiles_m <= 256))
    return launch_gemm_kblock(22, EPI == EPI_REQUANT, HAS_ZW, FAST, g, rq, dq, stream);
  // a few hundred activation rows against many channels: 256-channel x 128-row tiles keep the weight re-reads of
  // the square 128 tile away while still giving every CU a tile
  if (g.m <= 512 && (int64_t)((g.m + 127) / 128) * ((g.n + 255) / 256) >= 128)
    return launch_cfg<256, 128, EPI, HAS_ZW, FAST>(g, rq, dq, stream);
  // the 128 x 128 tile needs a quarter of the registers and 64 KiB of LDS: two workgroups share a CU, so one tile's
  // prologue and epilogue overlap the other's main loop (what short-K shapes are made of)
  // short K and more tiles than two per CU: three stages (48 KiB) let a third workgroup in, which saves a round of
  // tiles; the shallower prefetch only costs when K is long
  if (tiles_m > 512 && g.k <= 1024) return launch_cfg<128, 128, EPI, HAS_ZW, FAST, 3, 3>(g, rq, dq, stream);
  // short K, fp32 out and fewer 128 x 128 tiles than CUs: half-width tiles, three per CU, fill the device
  if (EPI == EPI_DEQUANT && tiles_m >= 128 && tiles_m < 256 && g.k <= 1024)
    return launch_cfg<64, 128, EPI, HAS_ZW, FAST, 4, 3>(g, rq, dq, stream);
  if (tiles_m >= 128) return launch_cfg<128, 128, EPI, HAS_ZW, FAST, 4, 2>(g, rq, dq, stream);
  // (what is left has few tiles of any size; with a long K the 64 x 64 tiles take eight stages as above)
  if (g.k_pad >= 1024) return launch_cfg<64, 64, EPI, HAS_ZW, FAST, 8, 2>(g, rq, dq, stream);
  return launch_cfg<64, 64, EPI, HAS_ZW, FAST>(g, rq, dq, stream);
}

// Large fp32 outputs are written with non-temporal stores: they are not re-read out of L2 by whatever runs next, and
// they do not queue behind dirty lines.  Measured over twelve shapes with 12-75 MB of output: 3-13 % faster (BERT QKV
// 22.0 -> 19.5 us) except where every tile of the grid finishes in the same moment (exactly three tiles per CU: 2-6 %
// slower), as long as rows are whole 128-byte lines: a line that two stores share is written to memory twice (4096 x 3070
// outputs 40.6 us, plain 21).  A compile-time choice: the two kinds of store under a run-time condition are merged into
// plain stores.
static bool stream_out_hint(int m, int n) { return (n & 31) == 0 && (int64_t)m * n * 4 >= ((int64_t)8 << 20); }

static int check_args(const int8_t *a, int64_t lda, int m, int k, const WeightView &wv, int n, const void *c,
                      int64_t ldc) {
  const int8_t *w = wv.w;
  const int k_pad = wv.k_pad;
  if (a == nullptr || w == nullptr || c == nullptr) {
    set_error("gemm: null pointer");
    return MI_NULL_PTR;
  }
  // (k_pad, ldw and ldc are not handed on: the kernels know them, see GemmCall)
  if (m <= 0 || n <= 0 || k <= 0 || (k & 15) != 0 || (lda & 15) != 0 || lda < k || lda > 0x7fffffff || k_pad != round_up(k, kKPad) ||
      wv.ldw != weight_row_stride(k_pad) || (reinterpret_cast<uintptr_t>(a) & 15) != 0 || ldc != n) {
    set_error("gemm: unsupported operand geometry m=%d n=%d k=%d lda=%lld k_pad=%d ldc=%lld", m, n, k, (long long)lda,
              k_pad, (long long)ldc);
    return MI_PARAM_INVALID;
  }
  return MI_OK;
}

int launch_gemm_requant(const int8_t *a, int64_t lda, int m, int k, const WeightView &w, int n,
                        const RequantParams &rq, int8_t *c, int64_t ldc, hipStream_t stream) {
  int rc = check_args(a, lda, m, k, w, n, c, ldc);
  if (rc != MI_OK) return rc;
  GemmArgs g{a, lda, m, k, w.w, w.ldw, w.k_pad, w.blocked, n, 0, 0, c, ldc};
  DequantParams dq{};
  if (rq.has_zw) {
    return rq.fast2 ? launch_pick_tile<EPI_REQUANT, true, true>(g, rq, dq, stream)
                    : launch_pick_tile<EPI_REQUANT, true, false>(g, rq, dq, stream);
  }
  return rq.fast2 ? launch_pick_tile<EPI_REQUANT, false, true>(g, rq, dq, stream)
                  : launch_pick_tile<EPI_REQUANT, false, false>(g, rq, dq, stream);
}

template <int TILE_N, int TILE_M, bool HAS_ZW, bool FAST, int NST, int OCC>
static int launch_conv_cfg(const ConvCall &call, hipStream_t stream) {
  auto kern = gemm_conv_kernel<TILE_N, TILE_M, HAS_ZW, FAST, NST, OCC>;
  launch_kernel(kern, dim3((call.m + TILE_M - 1) / TILE_M * ((call.n + TILE_N - 1) / TILE_N)), dim3(256), 0, stream, call);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <bool HAS_ZW, bool FAST>
static int launch_conv_pick_tile(const ConvCall &g, hipStream_t stream) {
  const int64_t tiles_m = (int64_t)((g.m + 127) / 128) * ((g.n + 127) / 128);
  // 64 x 64 tiles, four workgroups per CU (an allocation of 132 registers let in three, of which the second round was often
  // next to empty): a step's gathered loads take longer than its products, and what hides them is other workgroups.  us per
  // launch, three per CU / four: 8 x 28 x 28, 3x3, 96 -> 192 channels 11.0 / 7.4, 1x1 there 5.6 / 4.3; with few enough tiles for one
  // round of three no change (8 x 40 x 40, 48 -> 48 4.7; one 56 x 56 image, 64 -> 64 5.0).  64 x 128 tiles at 16 x 50 x 50,
  // 32 -> 32 5.9, these 5.7.
  // Up to 64 channels, 64 x 256 tiles, two per CU: the same number of pixels at once, weights read a quarter as often, but a
  // round of them (1024 rows of 128 pixels) is two of the small ones.  They win (a) where their last round is more than three
  // quarters full, unless the contraction is so short that prologue and stores are most of a tile, and (b) over several rounds
  // once the contraction pays for what the last one wastes.  us per launch, small /
  // tall, 64 -> 64 channels 3x3 (K = 576): 640 rows 10.4 / 12.0, 768 11.8 / 12.1, 800 13.0 / 12.2, 1024 14.8 / 13.5,
  // 1040 16.2 / 19.6, 1600 22.2 / 23.4, 2048 29.9 / 24.3, 3000 40.4 / 35.3; time of the tall ones relative to the small ones
  // at 1100 / 1400 / 1664 / 2300 / 3200 / 4300 rows: K = 288 1.19 1.05 1.06 1.04 1.03 0.91, with stride 2 1.27 1.12 1.11
  // 1.18 1.15 0.96, K = 576 1.13 1.00 1.01 1.00 0.88 0.86, stride 2 1.18 1.00 1.06 0.89 0.87 0.86, K = 864 1.08 0.93 0.91
  // 0.89 0.83 0.79, K = 144 1.28 1.12 1.16 1.15 1.15 1.09; (a) at 900 / 1950 rows: K = 144 0.99 1.05 (32 channels 0.92
  // 0.92), K = 288 0.98 0.93, stride 2 1.01 1.06, K = 576 0.89 0.88, stride 2 0.93 1.01; at 900 rows 1x1 with K = 64 1.08.
  // 128 x 128 tiles against more channels as soon as there are enough of them (32 x 28 x 28, 64 -> 128 7.2, on 64 x 64 9.1).
  const int64_t rows = (g.m + 127) / 128;
  const bool full_last_round = (rows - 1) % 1024 >= 768 && g.k >= (g.n <= 32 ? 144 : 288 * g.cv.stride_w);
  const bool many_rounds = rows >= 1400 && rows * g.k >= 1300000;
  if (g.n <= 64 && (full_last_round || many_rounds)) return launch_conv_cfg<64, 256, HAS_ZW, FAST, 4, 2>(g, stream);
  if (g.n > 64 && tiles_m >= 128) return launch_conv_cfg<128, 128, HAS_ZW, FAST, 4, 2>(g, stream);
  return launch_conv_cfg<64, 64, HAS_ZW, FAST, 4, 4>(g, stream);
}

bool gemm_conv_supported(const ConvGeom &cg, const void *in) {
  const int64_t k = (int64_t)cg.kernel_h * cg.kernel_w * cg.in_c;
  const auto fits = [](int x) { return x == (int16_t)x; };
  return fits(cg.stride_h) && fits(cg.stride_w) && fits(cg.dilation_h) && fits(cg.dilation_w) && fits(cg.pad_u) && fits(cg.pad_l) &&
         (cg.in_c & 15) == 0 && k <= 65536 - 128 && (int64_t)cg.in_h * cg.in_w * cg.in_c < ((int64_t)1 << 31) &&
         (int64_t)cg.batch * cg.out_h * cg.out_w < ((int64_t)1 << 31) && (reinterpret_cast<uintptr_t>(in) & 15) == 0;
}

int launch_gemm_conv_requant(const int8_t *in, const ConvGeom &cg, const int8_t *fill16, const WeightView &w,
                             const RequantParams &rq, int8_t *out, hipStream_t stream) {
  const int64_t k64 = (int64_t)cg.kernel_h * cg.kernel_w * cg.in_c;
  const int64_t m64 = (int64_t)cg.batch * cg.out_h * cg.out_w;
  if (in == nullptr || fill16 == nullptr || w.w == nullptr || out == nullptr) {
    set_error("gemm_conv: null pointer");
    return MI_NULL_PTR;
  }
  if (!gemm_conv_supported(cg, in) || m64 <= 0 || cg.out_c <= 0 || w.k_pad != round_up((int)k64, kKPad) ||
      w.ldw != weight_row_stride(w.k_pad)) {
    set_error("gemm_conv: unsupported geometry ic=%d k=%lld pixels=%lld oc=%d", cg.in_c, (long long)k64,
              (long long)m64, cg.out_c);
    return MI_PARAM_INVALID;
  }
  const auto magic = [](int d) { return d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + d - 1) / (uint64_t)d); };
  const ConvCall call{in, w.w, fill16, out, (int)m64, cg.out_c, (int)k64,
                      ConvGatherArgs{cg.in_h, cg.in_w, cg.in_c, cg.out_w, cg.out_h * cg.out_w, magic(cg.in_c), magic(cg.kernel_w),
                                     (int16_t)cg.stride_h, (int16_t)cg.stride_w, (int16_t)cg.dilation_h, (int16_t)cg.dilation_w,
                                     (int16_t)cg.pad_u, (int16_t)cg.pad_l, cg.kernel_w},
                      RequantCall::of(rq)};
  if (rq.has_zw) {
    return rq.fast2 ? launch_conv_pick_tile<true, true>(call, stream) : launch_conv_pick_tile<true, false>(call, stream);
  }
  return rq.fast2 ? launch_conv_pick_tile<false, true>(call, stream) : launch_conv_pick_tile<false, false>(call, stream);
}

int launch_gemm_dequant(const int8_t *a, int64_t lda, int m, int k, const WeightView &w, int n,
                        const DequantParams &dq, float *c, int64_t ldc, hipStream_t stream) {
  int rc = check_args(a, lda, m, k, w, n, c, ldc);
  if (rc != MI_OK) return rc;
  GemmArgs g{a, lda, m, k, w.w, w.ldw, w.k_pad, w.blocked, n, 0, 0, c, ldc};
  RequantParams rq{};
  // the third parameter (the fast-rounding switch of the int8 epilogue) selects non-temporal stores here
  const bool nt = stream_out_hint(m, n);
  if (dq.zw0 != 0) {
    return nt ? launch_pick_tile<EPI_DEQUANT, true, true>(g, rq, dq, stream)
              : launch_pick_tile<EPI_DEQUANT, true, false>(g, rq, dq, stream);
  }
  return nt ? launch_pick_tile<EPI_DEQUANT, false, true>(g, rq, dq, stream)
            : launch_pick_tile<EPI_DEQUANT, false, false>(g, rq, dq, stream);
}

// Rows that are no whole 16-byte chunks, or not aligned to them: the padded copy is a launch of its own, so where 64 x 64 tiles
// are the quickest they take the rows as they are, up to the K at which their unaligned loads, once per column tile, have
// cost as much.  us, copy and tiles / this: 333 x 1001 x 1000 7.4 / 5.6, 100 x 500 x 500 7.2 / 4.4, 128 x 768 x 770 7.5 / 5.7,
// 1000 x 1000 x 1001 8.0 / 6.8, 200 x 1000 x 1500 7.9 / 6.7, 200 x 1000 x 1793 8.5 / 9.2, x 2040 8.4 / 7.8, x 4003 12.5 / 16.5,
// 500 x 2000 x 3001 12.3 / 14.2; less than a block of 128: 65 x 120 x 64 6.4 / 3.9, 1000 x 65 x 1001 6.6 / 4.3, 200 x 17 x 4096
// 6.3 / 4.1, 8000 x 100 x 64 7.0 / 4.2.
constexpr int kAnyrowLeastK = 16, kAnyrowMostK = 1536;
static bool anyrow_tiles(int m, int k, int n) {
  if (k < kAnyrowLeastK || k > kAnyrowMostK) return false;
  float cost;
  const TileCost &t = cheapest_tile(m, k, 1, &n, &cost);
  return t.ring && t.tn == 1 && t.tm == 1;
}
static int short_any(int m, int k, int n, bool requant, bool short_form) {
  return short_form && k < (1 << 23) && short_goes_first(m, k) ? short_tile(m, k, n, requant).tile : 0;
}
static bool takes_any(int m, int k, const WeightView &w, int n, bool requant, bool short_form) {
  return w.blocked != nullptr && (anyrow_tiles(m, k, n) || short_any(m, k, n, requant, short_form) != 0);
}
static bool short_form(const RequantParams &rq, int, int) { return rq.fast2 != 0; }
static bool short_form(const DequantParams &, int m, int n) { return !stream_out_hint(m, n); }

bool gemm_anyrow_takes(int m, int k, const WeightView &w, int n, const RequantParams &rq) {
  return takes_any(m, k, w, n, true, short_form(rq, m, n));
}
bool gemm_anyrow_takes(int m, int k, const WeightView &w, int n, const DequantParams &dq) {
  return takes_any(m, k, w, n, false, short_form(dq, m, n));
}
bool gemm_short_takes(int m, int k, const WeightView &w, int n, const RequantParams &rq) {
  return w.blocked != nullptr && short_any(m, k, n, true, short_form(rq, m, n)) != 0;
}
bool gemm_short_takes(int m, int k, const WeightView &w, int n, const DequantParams &dq) {
  return w.blocked != nullptr && short_any(m, k, n, false, short_form(dq, m, n)) != 0;
}

static int launch_any_rows(bool requant, bool short_form, const int8_t *a, int m, int k, const WeightView &w, int n, const RequantParams &rq,
                           const DequantParams &dq, void *c, hipStream_t stream) {
  if (a == nullptr || c == nullptr) {
    set_error("gemm: null pointer");
    return MI_NULL_PTR;
  }
  if (m <= 0 || n <= 0 || !takes_any(m, k, w, n, requant, short_form) || w.k_pad != round_up(k, kKPad)) {
    set_error("gemm: unsupported operand geometry m=%d n=%d k=%d k_pad=%d", m, n, k, w.k_pad);
    return MI_PARAM_INVALID;
  }
  const GemmArgs g{a, k, m, k, nullptr, 0, w.k_pad, w.blocked, n, 0, 0, c, n};
  const bool has_zw = requant ? rq.has_zw != 0 : dq.zw0 != 0, any = (k & 15) != 0 || (reinterpret_cast<uintptr_t>(a) & 15) != 0;
  if (const int tile = short_any(m, k, n, requant, short_form)) return launch_gemm_short(tile, any, requant, has_zw, g, rq, dq, stream);
  return launch_gemm_anyrow(requant, has_zw, rq.fast2 != 0, g, rq, dq, stream);
}

int launch_gemm_anyrow_requant(const int8_t *a, int m, int k, const WeightView &w, int n, const RequantParams &rq, int8_t *c,
                               hipStream_t stream) {
  return launch_any_rows(true, short_form(rq, m, n), a, m, k, w, n, rq, DequantParams{}, c, stream);
}

int launch_gemm_anyrow_dequant(const int8_t *a, int m, int k, const WeightView &w, int n, const DequantParams &dq, float *c,
                               hipStream_t stream) {
  return launch_any_rows(false, short_form(dq, m, n), a, m, k, w, n, RequantParams{}, dq, c, stream);
}

// Several matrices against the same rows as one launch, where that is expected to take less than a launch each: a
// round of tiles more is the price of a launch that fills its last round badly, and there are fewer of those, on larger tiles.
// us per pair of 11008 x 4096, two launches -> one: int8 output, 128 rows 33.6 -> 26.3, 256 rows 47.6 -> 34.0, 512 rows
// 64.6 -> 51.5; fp32 output with a scale per row, 2048 rows 194.8 -> 181.
// The one launch is never split, so few channels of long K stay apart where each member alone is split.  kManyRows: per K block on
// 64 x 64 tiles of more rows than the weights stream past, which find them in the L2s.  us per pair (rows x channels x K), one
// launch / two split ones: 70 x 64 x 11008 25.7 / 16.05, 70 x 64 x 8192 18.75 / 14.8, 100 x 256 x 11008 21.95 / 17.5,
// 100 x 1024 x 11008 22.55 / 21.2, 128 x 512 x 8192 18.95 / 17.85, 200 x 64 x 16384 25.45 / 17.75, 512 x 128 x 32768 52.0 / 27.4; stay
// together: 128 x 512 x 7168 17.1 / 18.2, 100 x 1024 x 8192 16.95 / 18.2, 128 x 768 x 8192 19.15 / 18.65, 70 x 64 x 5120 13.45 / 14.3,
// 200 x 512 x 11008 19.55 / 21.0, 500 x 256 x 12288 20.0 / 21.4, three of 100 x 256 x 11008 26.3 / 26.3, four of 70 x 64 x 16384
// 35.95 / 36.3.
static const TileCost *group_tile(int64_t lda, int m, int k, int count, const WeightView *w, const int *n, bool requant, hipStream_t stream) {
  if (count < 2 || count > kGemmGroupMax || k < 1024 || !kblock_takes(k, lda)) return nullptr;
  float alone = 0.0f, alone_split = 0.0f, alone_unsplit = 0.0f, together;
  for (int i = 0; i < count; ++i) {
    if (w[i].blocked == nullptr || w[i].k_pad != w[0].k_pad) return nullptr;
    float cost;
    int parts;
    const TileCost &whole = cheapest_tile(m, k, 1, n + i, &cost);
    alone += cost;
    const ShortTile in_short = short_tile_of_chunks(m, k, n[i], requant);  // (the members' forms are those of gemm_short.hip and gemm_split.hip)
    alone_unsplit += in_short.tile != 0 ? in_short.cost : cost;
    if (in_short.tile != 0 && short_goes_first(m, k)) {
      cost = in_short.cost;
    } else {
      choose_split(m, k, n[i], whole, cost, &parts, &cost);
    }
    alone_split += cost;
  }
  const TileCost &t = cheapest_tile(m, k, count, n, &together);
  if (together >= alone) return nullptr;
  constexpr float kManyRows = 0.18f;
  if (t.ring && t.tn == 1 && t.tm == 1 && (m + 63) / 64 > kStreamRowTiles) together = t.a + kManyRows * (float)((k + 127) / 128);
  return together < (split_space(stream) != nullptr ? alone_split : alone_unsplit) ? &t : nullptr;
}

const TileCost *gemm_group_tile(int64_t lda, int m, int k, int count, const WeightView *w, const int *n, const RequantParams *rq,
                                hipStream_t stream) {
  for (int i = 0; i < count; ++i)
    if (rq[i].has_zw || !rq[i].fast2) return nullptr;
  return group_tile(lda, m, k, count, w, n, true, stream);
}

const TileCost *gemm_group_tile(int64_t lda, int m, int k, int count, const WeightView *w, const int *n, const DequantParams *dq,
                                hipStream_t stream) {
  for (int i = 0; i < count; ++i)
    if (dq[i].zw0 != 0) return nullptr;
  return group_tile(lda, m, k, count, w, n, false, stream);
}

template <typename P>
static int fill_group(const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w, const int *n, void *const *c,
                      const P *p, GemmGroup<P> *grp) {
  for (int i = 0; i < count; ++i) {
    const int rc = check_args(a, lda, m, k, w[i], n[i], c[i], n[i]);
    if (rc != MI_OK) return rc;
    grp->n[i] = n[i];
    grp->wb[i] = w[i].blocked;
    grp->c[i] = c[i];
    grp->p[i] = p[i];
  }
  grp->g = GemmArgs{a, lda, m, k, nullptr, 0, w[0].k_pad, nullptr, 0, 0, 0, nullptr, 0};
  grp->count = count;
  return MI_OK;
}

int launch_gemm_group_requant(const TileCost &t, const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w,
                              const int *n, const RequantParams *rq, int8_t *const *c, hipStream_t stream) {
  GemmGroup<RequantParams> grp{};
  const int rc = fill_group(a, lda, m, k, count, w, n, reinterpret_cast<void *const *>(c), rq, &grp);
  if (rc != MI_OK) return rc;
  return t.ring ? launch_gemm_ring_group(10 * t.tn + t.tm, grp, stream) : launch_gemm_kblock_group(10 * t.tn + t.tm, grp, stream);
}

int launch_gemm_group_dequant(const TileCost &t, const int8_t *a, int64_t lda, int m, int k, int count, const WeightView *w,
                              const int *n, const DequantParams *dq, float *const *c, hipStream_t stream) {
  GemmGroup<DequantParams> grp{};
  const int rc = fill_group(a, lda, m, k, count, w, n, reinterpret_cast<void *const *>(c), dq, &grp);
  if (rc != MI_OK) return rc;
  bool nt = true;
  for (int i = 0; i < count; ++i) nt = nt && stream_out_hint(m, n[i]);
  return t.ring ? launch_gemm_ring_group(10 * t.tn + t.tm, nt, grp, stream)
                : launch_gemm_kblock_group(10 * t.tn + t.tm, nt, grp, stream);
}

}  // namespace mi
