// The ring loop of gemm_ring.hip and gemm_split.hip.
#pragma once

#include "gemm_core.h"

namespace mi {

// Which part of a tile's K blocks a workgroup computes, and where the parts' sums meet (gemm_split.hip).
struct KPart {
  int part = 0, parts = 1;
  int tile = 0;                 // number of the tile
  int8_t *sums = nullptr;       // the parts' sums, tile by tile
  uint32_t *arrived = nullptr;  // per tile, zero between launches
};
template <int TN, int TM, bool HAS_ZW>
__device__ __forceinline__ bool add_parts(const KPart &kp, v16i (&acc)[TN][TM], int (&rowsum)[TM], int *lds, int tid);

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
// STREAM: weight loads carry the non-temporal hint (see kStreamRowTiles).
// SPLIT: the workgroup computes one of several parts of its tile's K blocks (see gemm_split.hip).
// =====================================================================================================================
template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST, bool STREAM, bool SPLIT = false>
__device__ __forceinline__ void gemm_ring_body(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, int tile_m,
                                               int tile_n, const KPart &kp = KPart()) {
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
  const int all_blocks = (g.k + KB - 1) / KB;
  // this workgroup's blocks: first_block + (0 .. last); `ends`: the last of them is K's last
  const int first_block = SPLIT ? kp.part * all_blocks / kp.parts : 0;
  const int last = (SPLIT ? (kp.part + 1) * all_blocks / kp.parts : all_blocks) - first_block - 1;
  const bool ends = !SPLIT || kp.part == kp.parts - 1;
  const int kchunks = g.k >> 4;
  EpiParams<TILE_N, EPI, FAST> epi;
  epi.fetch(rq, dq, n0, g.n, tid);
  DeqInput<TM> din;
  if (EPI == EPI_DEQUANT) din.fetch_rows(dq, m0 + wm * 32 * TM, r, g.m);

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
  const int a_last = (kchunks - 1) * 16 - (all_blocks - 1) * KB;  // offset of the last valid chunk in the last block
  auto a_offsets_for_last_block = [&]() {
    if (!ends) return;
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
                                                 blocked_weight_offset(wg.group(l >> 1), l & 1, k64, first_block + kb), 0, STREAM ? 2 : 0);
      } else {
        const int i = l - 2 * TN;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds_ptr(sa + i * 1024), 16, a_voff[i], (first_block + kb) * KB, 0, 0);
      }
    }
  };
  typedef std::integral_constant<int, 0> at0;
  typedef std::integral_constant<int, PART> at1;
  typedef std::integral_constant<int, LPB> at2;

  v16i acc[TN][TM];
  RowSums<TM> sums;
  if (HAS_ZW) sums.clear(lane);

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
  auto mma = [&](const Frag<TN, TM> &f, bool live) {  // live: the lane's 16 activation bytes lie inside K
    if (HAS_ZW) sums.add(f.a, live);
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
    constexpr int LOADS = decltype(loads_c)::value, MF = 2 * (TN + HAS_ZW) * TM, RD = 2 * (TN + TM);
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
  if (EPI == EPI_DEQUANT) din.fetch_tensor(dq);
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
    mma(fa[0], true);
    mma(fa[1], true);
    hints(std::integral_constant<int, LPB - PART>());
    // loads complete in order: blocks b + 2 .. b + S - 1 may still be on their way, block b + 1 is in
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * LPB) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (b + S == last) a_offsets_for_last_block();
    read_half(fa, next, 0);
    dma(st, b + S < last ? b + S : last, at0(), at1());  // (past the end: into a stage nobody reads any more)
    mma(fb[0], true);
    mma(fb[1], true);
    hints(std::integral_constant<int, PART>());
    advance();
  }
  while (b <= last) {  // the last blocks: nothing left to request
    read_half(fb, st, 1);
    mma(fa[0], (first_block + b) * 8 + h < kchunks);
    mma(fa[1], (first_block + b) * 8 + 2 + h < kchunks);
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
    mma(fb[0], (first_block + b) * 8 + 4 + h < kchunks);
    mma(fb[1], (first_block + b) * 8 + 6 + h < kchunks);
    hints(at0());
    advance();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every load has landed before the LDS is reused
  __syncthreads();
  int rowsum[TM] = {};
  if (HAS_ZW) sums.get(rowsum);
  if constexpr (SPLIT) {
    if (!add_parts<TN, TM, HAS_ZW>(kp, acc, rowsum, reinterpret_cast<int *>(lds), tid)) return;
  }
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

}  // namespace mi
