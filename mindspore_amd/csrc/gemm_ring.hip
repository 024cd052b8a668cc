// int8 GEMM on the matrix cores, K in blocks of 128 bytes through a ring of LDS stages (gemm_i8.hip says which shapes come
// here).
#include "gemm_core.h"

namespace mi {

// =====================================================================================================================
// The K blocks of gemm_kblock.hip through a ring of S LDS stages that hold both operands, S - 1 blocks ahead.
//
// A block of a tile smaller than 256 x 256 lasts 0.25 to 0.5 us on the matrix cores, and the fetch window of that loop
// (two blocks for W, one and a half for A) is then shorter than the way to memory and back: 192 x 128 tiles, one per CU,
// took 0.74 us a block for 0.38 us of MFMAs.  Where a CU has only one workgroup to run, the LDS that a second one would
// need holds further stages instead.  Everything else is as there: four quarters per block, double-buffered fragments,
// one barrier per block between quarter three and four; the loads of block b + S - 1 are spread over quarters 1 to 3 of
// block b and quarter 4 of the block before, which is the first moment its stage is free.
// Bound by the loads, where weights come from HBM: without its MFMAs the loop takes as long (512 x 12288 x 4096 29.8 of 30.1 us), with
// the weights in the caches 17; a CU gets 50 to 60 GB/s, whatever the number of CUs and of bytes in flight beyond 100 KiB, since
// its loads return in order, the activations' L2 hits behind the weights' misses.
// STREAM: weight loads carry the non-temporal hint (see launch_ring).
// =====================================================================================================================
template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST, bool STREAM>
__device__ __forceinline__ void gemm_ring_body(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, int tile_m,
                                               int tile_n) {
#if defined(__HIP_DEVICE_COMPILE__)  // the buffer-resource type exists in the device pass only; the host pass needs just the stub
  constexpr int TILE_N = 64 * TN, TILE_M = 64 * TM, KB = 128;
  constexpr int STAGE = (TILE_N + TILE_M) * KB;
  constexpr int LPB = 2 * (TN + TM);  // loader instructions per wave and block: 2 TN for W, then 2 TM for A
  constexpr int PART = LPB / 2;       // of which the second half of the block before issues this many
  static_assert(S >= 3, "at least two blocks ahead");
  static_assert(S * STAGE >= kEpiArrays * TILE_N * 4 + epi_wg_bytes<EPI, TN, TM>(), "the epilogue staging must fit");
  __shared__ __attribute__((aligned(1024))) char lds[S * STAGE];

  const int m0 = tile_m * TILE_M, n0 = tile_n * TILE_N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int r = lane & 31, h = lane >> 5;
  const int kblocks = (g.k + KB - 1) / KB, last = kblocks - 1;
  const int kchunks = g.k >> 4;
  EpiParams<TILE_N, EPI, FAST> epi;
  epi.fetch(rq, dq, n0, g.n, tid);
  DeqInput<TM> din;
  if (EPI == EPI_DEQUANT) din.fetch(dq, m0 + wm * 32 * TM, r, g.m);

  // loader.  W comes from the blocked copy: a wave takes TN groups of 16 channels, and an instruction fetches one 1 KiB
  // block (16 channels x 64 bytes of K, chunk by chunk: [chunk][channel]) front to back into the same order in LDS,
  // where 16 lanes of a fragment read then find 256 consecutive bytes.  A as in gemm_kblock_body.
  const int drow = lane >> 3;
  const int dchunk = (lane & 7) ^ (drow >> 1);  // for even i; odd i: ^ 4
  const int k64 = g.k_pad >> 6;
  const WaveWeightGroups<TN> wg(g.n, n0, wave, kNPad);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t *>(g.wb) + (int64_t)wg.first * k64 * 1024, (short)0, wg.inside * k64 * 1024, 0x00020000);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(g.a) + (int64_t)m0 * g.lda, (short)0, -1, 0x00020000);
  int a_voff[2 * TM];
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    int m = wave * 16 * TM + 8 * i + drow;
    m = m0 + m < g.m ? m : g.m - 1 - m0;
    a_voff[i] = m * (int)g.lda + ((dchunk ^ ((i & 1) << 2)) << 4);
  }
  const int a_last = (kchunks - 1) * 16 - last * KB;  // offset of the last valid chunk in the last block
  auto a_offsets_for_last_block = [&]() {
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) {
      const int c16 = (dchunk ^ ((i & 1) << 2)) << 4;
      a_voff[i] += (c16 < a_last ? c16 : a_last) - c16;
    }
  };
  auto lds_ptr = [](char *p) { return (__attribute__((address_space(3))) void *)p; };
  // loader instructions [from, to) of block kb into stage st
  auto dma = [&](int st, int kb, auto from_c, auto to_c) {
    constexpr int from = decltype(from_c)::value, to = decltype(to_c)::value;
    char *sw = lds + st * STAGE + wave * TN * 2048, *sa = lds + st * STAGE + TILE_N * KB + wave * 16 * TM * KB;
#pragma unroll
    for (int l = from; l < to; ++l) {
      if (l < 2 * TN) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, lds_ptr(sw + l * 1024), 16, lane * 16,
                                                 blocked_weight_offset(wg.group(l >> 1), l & 1, k64, kb), 0, STREAM ? 2 : 0);
      } else {
        const int i = l - 2 * TN;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds_ptr(sa + i * 1024), 16, a_voff[i], kb * KB, 0, 0);
      }
    }
  };
  typedef std::integral_constant<int, 0> at0;
  typedef std::integral_constant<int, PART> at1;
  typedef std::integral_constant<int, LPB> at2;

  v16i acc[TN][TM];
  int rowsum[TM];
#pragma unroll
  for (int j = 0; j < TM; ++j) rowsum[j] = 0;

  const int swz = (r >> 1) & 7;
  const int w_off = (wn * 2 * TN + (r >> 4)) * 2048 + h * 256 + (r & 15) * 16, a_off = TILE_N * KB + (wm * 32 * TM + r) * KB;
  Frag<TN, TM> fa[2], fb[2];
  auto read_half = [&](Frag<TN, TM> (&f)[2], int st, int half) {  // half: 64-byte half of the block
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const char *wb = lds + st * STAGE + w_off + half * 1024 + q * 512;
      const char *ab = lds + st * STAGE + a_off + (((4 * half + 2 * q + h) ^ swz) << 4);
#pragma unroll
      for (int i = 0; i < TN; ++i) f[q].w[i] = *reinterpret_cast<const v4i *>(wb + i * 4096);
#pragma unroll
      for (int j = 0; j < TM; ++j) f[q].a[j] = *reinterpret_cast<const v4i *>(ab + j * 32 * KB);
    }
  };
  auto mma = [&](const Frag<TN, TM> &f, int chunk) {
    if (HAS_ZW) {
      const int ones = chunk < kchunks ? 0x01010101 : 0;
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
      for (int jj = 0; jj < TM; ++jj) {
        const int j = (i & 1) ? TM - 1 - jj : jj;
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.w[i], f.a[j], acc[i][j], 0, 0, 0);
      }
  };
  // order of one half: the fragment reads behind the first MFMAs, the loads behind the others
  auto hints = [&](auto loads_c) {
    constexpr int LOADS = decltype(loads_c)::value, MF = 2 * TN * TM, RD = 2 * (TN + TM);
    constexpr int first = (MF + 1) / 2, rest = MF - first;
#pragma unroll
    for (int m = 0; m < first; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                         // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, (RD + first - 1) / first, 0);  // DS read
    }
#pragma unroll
    for (int m = 0; m < rest; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if constexpr (LOADS > 0) __builtin_amdgcn_sched_group_barrier(0x020, (LOADS + rest - 1) / rest, 0);  // global -> LDS
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  if (last < S - 1) {
    for (int b = 0; b < last; ++b) dma(b, b, at0(), at2());
    a_offsets_for_last_block();
    dma(last, last, at0(), at2());
  } else {
#pragma unroll
    for (int b = 0; b < S - 1; ++b) dma(b, b, at0(), at2());
    if (last == S - 1) a_offsets_for_last_block();
    dma(S - 1, S - 1, at0(), at1());
  }
  // the accumulator registers are set while the first tiles are on their way
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = (int)kAccBias;
  if (last < S - 1) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 2) * LPB + PART) : "memory");  // block 0 is in
  }
  read_half(fa, 0, 0);
  int st = 0, prev = S - 1, next = 1, b = 0;  // stages of blocks b, b - 1 (and so b + S - 1), b + 1
  auto advance = [&]() {
    prev = st;
    st = next;
    next = next + 1 == S ? 0 : next + 1;
    ++b;
  };
  while (b + S - 1 <= last) {
    read_half(fb, st, 1);
    dma(prev, b + S - 1, at1(), at2());
    mma(fa[0], b * 8 + h);
    mma(fa[1], b * 8 + 2 + h);
    hints(std::integral_constant<int, LPB - PART>());
    // loads complete in order: blocks b + 2 .. b + S - 1 may still be on their way, block b + 1 is in
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * LPB) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (b + S == last) a_offsets_for_last_block();
    read_half(fa, next, 0);
    dma(st, b + S < last ? b + S : last, at0(), at1());  // (past the end: into a stage nobody reads any more)
    mma(fb[0], b * 8 + 4 + h);
    mma(fb[1], b * 8 + 6 + h);
    hints(std::integral_constant<int, PART>());
    advance();
  }
  while (b <= last) {  // the last blocks: nothing left to request
    read_half(fb, st, 1);
    mma(fa[0], b * 8 + h);
    mma(fa[1], b * 8 + 2 + h);
    hints(at0());
    const int later = last - b - 1;  // blocks behind b + 1 that may still be on their way
    if (S > 3 && later >= 2) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S > 3 ? 2 : 0) * LPB + PART) : "memory");
    } else if (later == 1) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LPB + PART) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PART) : "memory");
    }
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read_half(fa, next, 0);  // (behind the last block: bytes nobody uses)
    mma(fb[0], b * 8 + 4 + h);
    mma(fb[1], b * 8 + 6 + h);
    hints(at0());
    advance();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every load has landed before the LDS is reused
  __syncthreads();
  epi.to_lds(reinterpret_cast<int *>(lds), tid);
  gemm_epilogue<TILE_N, TN, TM, EPI, HAS_ZW, FAST, kAccBias, true>(
      acc, rowsum, g, rq, dq, din, reinterpret_cast<const int *>(lds),
      lds + kEpiArrays * TILE_N * 4 + wave * epi_stage_bytes<EPI, TM>(), lds + kEpiArrays * TILE_N * 4, n0, m0,
      n0 + wn * 32 * TN, m0 + wm * 32 * TM, r, h);
#endif
}

template <int TN, int TM, int S>
constexpr int ring_occupancy() {
  return 8 * (TN + TM) * S * 2 <= 160 ? 2 : 1;
}

template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST, bool STREAM>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(ring_occupancy<TN, TM, S>(), ring_occupancy<TN, TM, S>()))) void gemm_ring_kernel(
        GemmCall<EPI> call) {
  GemmArgs g;
  RequantParams rq;
  DequantParams dq;
  call.open(&g, &rq, &dq);
  int tile_m, tile_n;
  tile_coords(g, &tile_m, &tile_n);
  gemm_ring_body<TN, TM, S, EPI, HAS_ZW, FAST, STREAM>(g, rq, dq, tile_m, tile_n);
}

template <int TN, int TM, int S, bool STREAM>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(ring_occupancy<TN, TM, S>(), ring_occupancy<TN, TM, S>()))) void gemm_ring_group_kernel(
        GemmGroup<RequantParams> grp) {
  int tile_m, tile_n;
  tile_coords(grp.g, &tile_m, &tile_n);
  GemmArgs g;
  RequantParams rq;
  pick_member(grp, &tile_n, &g, &rq);
  gemm_ring_body<TN, TM, S, EPI_REQUANT, false, true, STREAM>(g, rq, DequantParams{}, tile_m, tile_n);
}

template <int TN, int TM, int S, bool FAST, bool STREAM>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(ring_occupancy<TN, TM, S>(), ring_occupancy<TN, TM, S>()))) void gemm_ring_group_deq_kernel(
        GemmGroup<DequantParams> grp) {
  int tile_m, tile_n;
  tile_coords(grp.g, &tile_m, &tile_n);
  GemmArgs g;
  DequantParams dq;
  pick_member(grp, &tile_n, &g, &dq);
  gemm_ring_body<TN, TM, S, EPI_DEQUANT, false, FAST, STREAM>(g, RequantParams{}, dq, tile_m, tile_n);
}

// Up to two row tiles the weights stream past the L2s, which then keep the activations that every channel tile re-reads.  With
// more row tiles too many workgroups rely on finding them there.  us per launch, weights from HBM, plain -> streamed: one row
// tile, 128 x 12288 x 4096 18.4 -> 16.3, 128 x 11008 x 4096 17.6 -> 16.0; two, 256 x 12288 x 4096 26.3 -> 23.4,
// 128 x 4096 x 4096 11.8 -> 11.0; three, 300 x 5504 x 2048 (fp32) 13.9 -> 14.8; four, 197 x 768 x 3072 (fp32) 8.2 -> 9.4;
// thirty-two, 4096 x 768 x 3072 (fp32) 16.3 -> 22.0.
constexpr int kStreamRowTiles = 2;

template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST>
static int launch_ring(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  const auto call = GemmCall<EPI>::of(g, g.wb, 64 * TN, 64 * TM, rq, dq);
  if (call.tiles_m <= kStreamRowTiles) {
    hipLaunchKernelGGL((gemm_ring_kernel<TN, TM, S, EPI, HAS_ZW, FAST, true>), call.grid(), dim3(256), 0, stream, call);
  } else {
    hipLaunchKernelGGL((gemm_ring_kernel<TN, TM, S, EPI, HAS_ZW, FAST, false>), call.grid(), dim3(256), 0, stream, call);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int TN, int TM, int S>
static int with_form(bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                     hipStream_t stream) {
  if (requant && has_zw == true && fast == true) return launch_ring<TN, TM, S, EPI_REQUANT, true, true>(g, rq, dq, stream);
  if (requant && has_zw == true && fast == false) return launch_ring<TN, TM, S, EPI_REQUANT, true, false>(g, rq, dq, stream);
  if (requant && has_zw == false && fast == true) return launch_ring<TN, TM, S, EPI_REQUANT, false, true>(g, rq, dq, stream);
  if (requant && has_zw == false && fast == false) return launch_ring<TN, TM, S, EPI_REQUANT, false, false>(g, rq, dq, stream);
  if (!requant && has_zw == true && fast == true) return launch_ring<TN, TM, S, EPI_DEQUANT, true, true>(g, rq, dq, stream);
  if (!requant && has_zw == true && fast == false) return launch_ring<TN, TM, S, EPI_DEQUANT, true, false>(g, rq, dq, stream);
  if (!requant && has_zw == false && fast == true) return launch_ring<TN, TM, S, EPI_DEQUANT, false, true>(g, rq, dq, stream);
  if (!requant && has_zw == false && fast == false) return launch_ring<TN, TM, S, EPI_DEQUANT, false, false>(g, rq, dq, stream);
  return MI_ERROR;
}

int launch_gemm_ring(int tile, bool requant, bool has_zw, bool fast, GemmArgs g, const RequantParams &rq,
                     const DequantParams &dq, hipStream_t stream) {
  if (g.wb == nullptr) {
    set_error("gemm: the blocked weight copy is missing");
    return MI_NULL_PTR;
  }
  switch (tile) {  // as many stages as the LDS of a CU holds (1 x 1: of half a CU)
    case 11: return with_form<1, 1, 5>(requant, has_zw, fast, g, rq, dq, stream);
    case 12: return with_form<1, 2, 6>(requant, has_zw, fast, g, rq, dq, stream);
    case 22: return with_form<2, 2, 5>(requant, has_zw, fast, g, rq, dq, stream);
    case 32: return with_form<3, 2, 4>(requant, has_zw, fast, g, rq, dq, stream);
    case 24: return with_form<2, 4, 3>(requant, has_zw, fast, g, rq, dq, stream);
    case 42: return with_form<4, 2, 3>(requant, has_zw, fast, g, rq, dq, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

template <int TN, int TM, int S>
static int launch_group(GemmGroup<RequantParams> grp, hipStream_t stream) {
  const dim3 grid(group_tiles(&grp, 64 * TN, 64 * TM));
  if (grp.g.tiles_m <= kStreamRowTiles) {
    hipLaunchKernelGGL((gemm_ring_group_kernel<TN, TM, S, true>), grid, dim3(256), 0, stream, grp);
  } else {
    hipLaunchKernelGGL((gemm_ring_group_kernel<TN, TM, S, false>), grid, dim3(256), 0, stream, grp);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int TN, int TM, int S, bool FAST>
static int launch_group_deq(GemmGroup<DequantParams> grp, hipStream_t stream) {
  const dim3 grid(group_tiles(&grp, 64 * TN, 64 * TM));
  if (grp.g.tiles_m <= kStreamRowTiles) {
    hipLaunchKernelGGL((gemm_ring_group_deq_kernel<TN, TM, S, FAST, true>), grid, dim3(256), 0, stream, grp);
  } else {
    hipLaunchKernelGGL((gemm_ring_group_deq_kernel<TN, TM, S, FAST, false>), grid, dim3(256), 0, stream, grp);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

int launch_gemm_ring_group(int tile, GemmGroup<RequantParams> grp, hipStream_t stream) {
  switch (tile) {
    case 11: return launch_group<1, 1, 5>(grp, stream);
    case 12: return launch_group<1, 2, 6>(grp, stream);
    case 22: return launch_group<2, 2, 5>(grp, stream);
    case 32: return launch_group<3, 2, 4>(grp, stream);
    case 24: return launch_group<2, 4, 3>(grp, stream);
    case 42: return launch_group<4, 2, 3>(grp, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

int launch_gemm_ring_group(int tile, bool fast, GemmGroup<DequantParams> grp, hipStream_t stream) {
  switch (tile) {
    case 11: return fast ? launch_group_deq<1, 1, 5, true>(grp, stream) : launch_group_deq<1, 1, 5, false>(grp, stream);
    case 12: return fast ? launch_group_deq<1, 2, 6, true>(grp, stream) : launch_group_deq<1, 2, 6, false>(grp, stream);
    case 22: return fast ? launch_group_deq<2, 2, 5, true>(grp, stream) : launch_group_deq<2, 2, 5, false>(grp, stream);
    case 32: return fast ? launch_group_deq<3, 2, 4, true>(grp, stream) : launch_group_deq<3, 2, 4, false>(grp, stream);
    case 24: return fast ? launch_group_deq<2, 4, 3, true>(grp, stream) : launch_group_deq<2, 4, 3, false>(grp, stream);
    case 42: return fast ? launch_group_deq<4, 2, 3, true>(grp, stream) : launch_group_deq<4, 2, 3, false>(grp, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

}  // namespace mi
