// int8 GEMM on the matrix cores, K in blocks of 128 bytes through five LDS slots (gemm_i8.hip says which shapes come here).
#include "gemm_core.h"

namespace mi {

// =====================================================================================================================
// K-block main loop for the 256 x 256 tile (one workgroup per CU, the whole register file).
//
// What the compute-bound GEMM pays for is operand delivery: the L2 -> L1 path moves whole 128-byte lines, so a loader
// that asks for 64 bytes of a row per K step has every line sent twice, one K step apart.  Here K advances in blocks of 128 bytes
// -- whole cache lines -- so that each line leaves the L2 once: one wave instruction fetches 8 rows x 128 bytes.
// LDS holds three slots for W and two for A (slot = 256 rows x 128 B = 32 KiB; all 160 KiB of the CU).  The path from
// the L1 into LDS moves 64 bytes per clock and CU: four waves issuing eight 1 KiB loads each within one quarter of a
// block saturate it, and a wave whose load does not fit the queue cannot issue its next MFMA either.  So every quarter
// issues four loads per wave, which takes a load window of a whole block per operand, hence the third W slot.  A loop
// iteration is one K block = four 32-byte MFMA sub-steps (quarters) on double-buffered fragments:
//   Q1  MFMAs on chunks 0-1 | reads chunks 2-3 | loads the second half of A block b+1
//   Q2  MFMAs on chunks 2-3 | reads chunks 4-5 | loads the first half of W block b+2 (into block b-1's slot)
//   Q3  MFMAs on chunks 4-5 | reads chunks 6-7 | loads the second half of W block b+2, then waits until all but
//       these eight W loads have landed (loads complete in order) and meets the other waves: block b+1 is complete
//       in LDS and nobody reads block b any more
//   Q4  MFMAs on chunks 6-7 | reads chunks 0-1 of block b+1 | loads the first half of A block b+2 into block b's slot
// One barrier per 128 bytes of K.  In a slot, 16-byte chunk c of row R sits at position c ^ ((R >> 1) & 7): the LDS
// has 64 banks (256 bytes per clock), so 16 consecutive rows of one logical chunk -- what 16 lanes of a fragment
// read ask for -- must land on 16 different 16-byte positions of a 256-byte period, and two rows of 128 bytes make
// one period.
//
// kAccBias: the accumulators start from this constant instead of 0 and the epilogue's per-channel constants take it
// out again (exact: wrap-around arithmetic).  Partial sums of signed products hover around zero, where every sign
// change flips all upper bits of the 32-bit accumulator; from an alternating bit pattern a sum that crosses it
// flips at most the bits up to the next 0/1 boundary.  The matrix pipe alone, on operands drawn like this
// benchmark's, sustains 7-9 % more (power-limited shader clock) with it.  For the same reason consecutive MFMAs
// share one operand (serpentine order over the 4 x 4 sub-tiles): +5 %.
// =====================================================================================================================
// TN x TM: the wave's sub-tile in MFMA tiles of 32 channels x 32 rows; the workgroup's tile is 64 TN channels x 64 TM
// rows, its W slots are TN x 8 KiB, its A slots TM x 8 KiB.  4 x 4 is the 256 x 256 tile described above; per quarter a
// wave has TN x TM MFMAs, TN + TM fragment reads and TN or TM loads.  2 x 2 (80 KiB of LDS, a quarter of the registers)
// lets two workgroups share a CU: for shapes with fewer than one 256 x 256 tile per CU, or short K, where one tile's
// prologue and epilogue have to overlap another tile's main loop.
// WB: W comes from the blocked copy of the weights, 1 KiB (16 channels x 64 bytes of K) front to back per instruction and in
// that order into LDS, where 16 lanes of a fragment read find 256 consecutive bytes; weights that have to come from HBM
// arrive sooner that way than as 128-byte pieces of 8 rows (2048 x 4096 x 11008 93 -> 88 us; handles without the blocked
// copy, and convolutions, read the row-major one).
template <int TN, int TM, int EPI, bool HAS_ZW, bool FAST, bool WB>
__device__ __forceinline__ void gemm_kblock_body(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, int tile_m,
                                                 int tile_n) {
#if defined(__HIP_DEVICE_COMPILE__)  // the buffer-resource type exists in the device pass only; the host pass needs just the stub
  constexpr int TILE_N = 64 * TN, TILE_M = 64 * TM, KB = 128;
  constexpr int SLOT_W = TILE_N * KB, SLOT_A = TILE_M * KB;
  constexpr int LDS_BYTES = 3 * SLOT_W + 2 * SLOT_A;  // W slots 0-2, A slots 0-1
  static_assert(LDS_BYTES >= kEpiArrays * TILE_N * 4 + epi_wg_bytes<EPI, TN, TM>(), "the epilogue staging must fit");
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];

  const int m0 = tile_m * TILE_M, n0 = tile_n * TILE_N;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int r = lane & 31, h = lane >> 5;
  const int kblocks = (g.k + KB - 1) / KB;
  const int kchunks = g.k >> 4;
  EpiParams<TILE_N, EPI, FAST> epi;
  epi.fetch(rq, dq, n0, g.n, tid);
  DeqInput<TM> din;
  if (EPI == EPI_DEQUANT) din.fetch_rows(dq, m0 + wm * 32 * TM, r, g.m);

  // loader: a wave fills a quarter of each slot, 16 T rows, 8 per instruction: instruction i takes rows
  // 16 T * wave + 8 * i + (lane >> 3); lane L writes position L & 7 of its row, i.e. fetches logical chunk
  // (L & 7) ^ ((row >> 1) & 7).  The loads are buffer loads: the address is descriptor base + per-lane byte offset (a
  // loop constant) + a scalar offset (row group and K block), so issuing one costs scalar instructions only.
  const int drow = lane >> 3;
  const int dchunk = (lane & 7) ^ (drow >> 1);  // for even i; odd i: ^ 4
  const int k64 = g.k_pad >> 6;
  const WaveWeightGroups<TN> wg(g.n, n0, wave, kNPad);
  const int64_t group_bytes = WB ? k64 * 1024 : 16 * g.ldw;
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t *>(WB ? g.wb : g.w) + wg.first * group_bytes, (short)0,
      wg.inside * (int)group_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(g.a) + (int64_t)m0 * g.lda, (short)0, -1, 0x00020000);
  // row-major: ldw is a multiple of 256, so odd i is w_voff ^ 64
  const int w_voff = WB ? lane * 16 : drow * g.ldw + dchunk * 16;
  int a_voff[2 * TM];
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    int m = wave * 16 * TM + 8 * i + drow;
    m = m0 + m < g.m ? m : g.m - 1 - m0;
    a_voff[i] = m * (int)g.lda + ((dchunk ^ ((i & 1) << 2)) << 4);
  }
  // A has exactly K valid bytes per row (the weights are zero padded, A is the caller's): in the last K block a
  // 16-byte chunk past K is fetched from the row's last chunk instead.  The offsets are moved there once, before
  // that block is first requested (in the 256 x 256 form the re-fetches after it ask for the same block).
  const int a_last = (kchunks - 1) * 16 - (kblocks - 1) * KB;  // offset of the last valid chunk in the last block
  auto a_offsets_for_last_block = [&]() {
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) {
      const int c16 = (dchunk ^ ((i & 1) << 2)) << 4;
      a_voff[i] += (c16 < a_last ? c16 : a_last) - c16;
    }
  };
  auto lds_ptr = [](char *p) { return (__attribute__((address_space(3))) void *)p; };
  // half: 0 = the first half of the wave's loader instructions (the upper half of its rows), 1 = the other half
  auto dma_w = [&](int slot, int kb, int half) {
    char *dst = lds + slot * SLOT_W + wave * 16 * TN * KB;
#pragma unroll
    for (int ii = 0; ii < TN; ++ii) {
      const int i = half * TN + ii;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, lds_ptr(dst + i * 1024), 16, WB ? w_voff : w_voff ^ ((i & 1) << 6),
                                               WB ? blocked_weight_offset(wg.group(i >> 1), i & 1, k64, kb)
                                                  : row_major_weight_offset(wg.group(i >> 1), i & 1, g.ldw, kb), 0, 0);
    }
  };
  auto dma_a = [&](int slot, int kb, int half) {
    char *dst = lds + 3 * SLOT_W + slot * SLOT_A + wave * 16 * TM * KB;
#pragma unroll
    for (int ii = 0; ii < TM; ++ii) {
      const int i = half * TM + ii;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds_ptr(dst + i * 1024), 16, a_voff[i], kb * KB, 0, 0);
    }
  };

  v16i acc[TN][TM];
  int rowsum[TM];
#pragma unroll
  for (int j = 0; j < TM; ++j) rowsum[j] = 0;
  // the accumulator registers are set while the first tiles are on their way (see below)
  auto init_accumulators = [&]() {
    const int bias = (int)kAccBias;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e)  // volatile: stays ahead of the wait for the first tiles
          asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(acc[i][j][e]) : "v"(bias));
  };

  const int swz = (r >> 1) & 7;
  const int w_off = WB ? (wn * 2 * TN + (r >> 4)) * 2048 + h * 256 + (r & 15) * 16 : (wn * 32 * TN + r) * KB;
  const int a_off = 3 * SLOT_W + (wm * 32 * TM + r) * KB;
  Frag<TN, TM> f0, f1;
  auto read_frag = [&](Frag<TN, TM> &f, int wslot, int aslot, int q) {  // q: 32-byte sub-step inside the block
    const int c = ((2 * q + h) ^ swz) << 4;
    const char *wb = lds + wslot * SLOT_W + w_off + (WB ? (q >> 1) * 1024 + (q & 1) * 512 : c);
    const char *ab = lds + aslot * SLOT_A + a_off + c;
#pragma unroll
    for (int i = 0; i < TN; ++i) f.w[i] = *reinterpret_cast<const v4i *>(wb + i * 32 * KB);
#pragma unroll
    for (int j = 0; j < TM; ++j) f.a[j] = *reinterpret_cast<const v4i *>(ab + j * 32 * KB);
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
  // Order of one quarter with LOADS loader instructions.  Where there are MFMAs enough: an LDS read behind each of the
  // first, then a load behind every other (4 x 4) or every one of the rest; otherwise LOADS groups of MFMAs, each with
  // its share of the reads and one load at its end.
  auto hints = [&](auto loads_c) {
    constexpr int LOADS = decltype(loads_c)::value, MF = TN * TM, RD = TN + TM;
    if constexpr (MF >= RD + LOADS) {
      constexpr int per = (MF - RD) / LOADS > 1 ? 2 : 1;
#pragma unroll
      for (int i = 0; i < RD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
      }
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, per, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);    // global -> LDS load issue
      }
    } else {
      constexpr int group = MF / LOADS > 0 ? MF / LOADS : 1, reads = (RD + MF - 1) / MF;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
#pragma unroll
        for (int m = 0; m < group; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  typedef std::integral_constant<int, TN> loads_w;
  typedef std::integral_constant<int, TM> loads_a;

  const int last = kblocks - 1;
  if (kblocks == 1) a_offsets_for_last_block();
  dma_w(0, 0, 0);
  dma_w(0, 0, 1);
  dma_a(0, 0, 0);
  dma_a(0, 0, 1);
  if (kblocks == 2) a_offsets_for_last_block();
  dma_w(1, last < 1 ? last : 1, 0);
  dma_w(1, last < 1 ? last : 1, 1);
  dma_a(1, last < 1 ? last : 1, 0);
  if (EPI == EPI_DEQUANT) din.fetch_tensor(dq);
  init_accumulators();
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * TN + TM) : "memory");  // W(0) and A(0) are in
  read_frag(f0, 0, 0, 0);
  int ws = 0, ws1 = 1, ws2 = 2;  // W slots of blocks b, b+1, b+2
  auto k_block_clamped = [&](int b) {
    const int as = b & 1;
    const int kb1 = b + 1 < last ? b + 1 : last;  // past the end: the last block again, into a slot nobody reads
    const int kb2 = b + 2 < last ? b + 2 : last;
    read_frag(f1, ws, as, 1);
    dma_a(as ^ 1, kb1, 1);
    mma(f0, b * 8 + h);
    hints(loads_a());
    read_frag(f0, ws, as, 2);
    dma_w(ws2, kb2, 0);
    mma(f1, b * 8 + 2 + h);
    hints(loads_w());
    read_frag(f1, ws, as, 3);
    dma_w(ws2, kb2, 1);
    mma(f0, b * 8 + 4 + h);
    hints(loads_w());
    // everything but the loads of W block b+2 has landed: that includes all of block b+1
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * TN) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (b + 3 == kblocks) a_offsets_for_last_block();
    read_frag(f0, ws1, as ^ 1, 0);
    dma_a(as, kb2, 0);
    mma(f1, b * 8 + 6 + h);
    hints(loads_a());
    const int t = ws;
    ws = ws1;
    ws1 = ws2;
    ws2 = t;
  };
  // One K block.  NEXT1 / NEXT2: blocks b + 1 / b + 2 exist.  The last two blocks have their own copies of the body
  // without the loads for blocks that do not exist (with 6 K blocks those would be a third of the operand traffic),
  // and the last one also without the barrier and the read-ahead.
  auto k_block = [&](int b, auto next1_c, auto next2_c) {
    constexpr bool NEXT1 = decltype(next1_c)::value, NEXT2 = decltype(next2_c)::value;
    const int as = b & 1;
    read_frag(f1, ws, as, 1);
    if (NEXT1) dma_a(as ^ 1, b + 1, 1);
    mma(f0, b * 8 + h);
    hints(loads_a());
    read_frag(f0, ws, as, 2);
    if (NEXT2) dma_w(ws2, b + 2, 0);
    mma(f1, b * 8 + 2 + h);
    hints(loads_w());
    read_frag(f1, ws, as, 3);
    if (NEXT2) dma_w(ws2, b + 2, 1);
    mma(f0, b * 8 + 4 + h);
    hints(loads_w());
    if (NEXT2) {
      // everything but the loads of W block b+2 has landed: that includes all of block b+1
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * TN) : "memory");
    } else if (NEXT1) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // block b+1, the last one, is in
    }
    __builtin_amdgcn_sched_barrier(0);
    if (NEXT2 && b + 3 == kblocks) a_offsets_for_last_block();
    if (NEXT1) read_frag(f0, ws1, as ^ 1, 0);
    if (NEXT2) dma_a(as, b + 2, 0);
    mma(f1, b * 8 + 6 + h);
    hints(loads_a());
    const int t = ws;
    ws = ws1;
    ws1 = ws2;
    ws2 = t;
  };
  if constexpr (TN < 4 || TM < 4) {
    for (int b = 0; b + 2 < kblocks; ++b) k_block(b, std::true_type(), std::true_type());
    if (kblocks >= 2) k_block(last - 1, std::true_type(), std::false_type());
    k_block(last, std::false_type(), std::false_type());
  } else {
    // (three copies of the 64-MFMA body push the 256 x 256 tile's register allocation into spilling, and at its
    //  K the two blocks' worth of extra loads are a few per cent: it keeps one body and lets the loads past the
    //  end fetch the last block again, into slots nobody reads)
    for (int b = 0; b < kblocks; ++b) k_block_clamped(b);
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

// workgroups per CU that the LDS leaves room for (and the register allocation is told to)
template <int TN, int TM>
constexpr int kblock_occupancy() {
  return (24 * TN + 16 * TM) * 2 <= 160 ? 2 : 1;
}

template <int TN, int TM, int EPI, bool HAS_ZW, bool FAST, bool WB>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(kblock_occupancy<TN, TM>(), kblock_occupancy<TN, TM>()))) void gemm_kblock_kernel(
        GemmCall<EPI> call) {
  GemmArgs g;
  RequantParams rq;
  DequantParams dq;
  call.open(&g, &rq, &dq);
  int tile_m, tile_n;
  tile_coords(g, &tile_m, &tile_n);
  gemm_kblock_body<TN, TM, EPI, HAS_ZW, FAST, WB>(g, rq, dq, tile_m, tile_n);
}

template <int TN, int TM>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(kblock_occupancy<TN, TM>(), kblock_occupancy<TN, TM>()))) void gemm_kblock_group_kernel(
        GemmGroup<RequantParams> grp) {
  int tile_m, tile_n;
  tile_coords(grp.g, &tile_m, &tile_n);
  GemmArgs g;
  RequantParams rq;
  pick_member(grp, &tile_n, &g, &rq);
  gemm_kblock_body<TN, TM, EPI_REQUANT, false, true, true>(g, rq, DequantParams{}, tile_m, tile_n);
}

template <int TN, int TM, bool FAST>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(kblock_occupancy<TN, TM>(), kblock_occupancy<TN, TM>()))) void gemm_kblock_group_deq_kernel(
        GemmGroup<DequantParams> grp) {
  int tile_m, tile_n;
  tile_coords(grp.g, &tile_m, &tile_n);
  GemmArgs g;
  DequantParams dq;
  pick_member(grp, &tile_n, &g, &dq);
  gemm_kblock_body<TN, TM, EPI_DEQUANT, false, FAST, true>(g, RequantParams{}, dq, tile_m, tile_n);
}

template <int TN, int TM, int EPI, bool HAS_ZW, bool FAST>
static int launch_kblock(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  const auto call = GemmCall<EPI>::of(g, g.wb != nullptr ? g.wb : g.w, 64 * TN, 64 * TM, rq, dq);
  if (g.wb != nullptr) {
    launch_kernel((gemm_kblock_kernel<TN, TM, EPI, HAS_ZW, FAST, true>), call.grid(), dim3(256), 0, stream, call);
  } else if constexpr (TN == TM) {
    launch_kernel((gemm_kblock_kernel<TN, TM, EPI, HAS_ZW, FAST, false>), call.grid(), dim3(256), 0, stream, call);
  } else {  // (rectangular tiles are chosen for the blocked copy only)
    set_error("gemm: the blocked weight copy is missing");
    return MI_NULL_PTR;
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int TN, int TM>
static int with_form(bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                     hipStream_t stream) {
  if (requant && has_zw == true && fast == true) return launch_kblock<TN, TM, EPI_REQUANT, true, true>(g, rq, dq, stream);
  if (requant && has_zw == true && fast == false) return launch_kblock<TN, TM, EPI_REQUANT, true, false>(g, rq, dq, stream);
  if (requant && has_zw == false && fast == true) return launch_kblock<TN, TM, EPI_REQUANT, false, true>(g, rq, dq, stream);
  if (requant && has_zw == false && fast == false) return launch_kblock<TN, TM, EPI_REQUANT, false, false>(g, rq, dq, stream);
  if (!requant && has_zw == true && fast == true) return launch_kblock<TN, TM, EPI_DEQUANT, true, true>(g, rq, dq, stream);
  if (!requant && has_zw == true && fast == false) return launch_kblock<TN, TM, EPI_DEQUANT, true, false>(g, rq, dq, stream);
  if (!requant && has_zw == false && fast == true) return launch_kblock<TN, TM, EPI_DEQUANT, false, true>(g, rq, dq, stream);
  if (!requant && has_zw == false && fast == false) return launch_kblock<TN, TM, EPI_DEQUANT, false, false>(g, rq, dq, stream);
  return MI_ERROR;
}

int launch_gemm_kblock(int tile, bool requant, bool has_zw, bool fast, GemmArgs g, const RequantParams &rq,
                       const DequantParams &dq, hipStream_t stream) {
  switch (tile) {
    case 44: return with_form<4, 4>(requant, has_zw, fast, g, rq, dq, stream);
    case 34: return with_form<3, 4>(requant, has_zw, fast, g, rq, dq, stream);
    case 22: return with_form<2, 2>(requant, has_zw, fast, g, rq, dq, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

template <int TN, int TM>
static int launch_group(GemmGroup<RequantParams> grp, hipStream_t stream) {
  const dim3 grid(group_tiles(&grp, 64 * TN, 64 * TM));
  launch_kernel((gemm_kblock_group_kernel<TN, TM>), grid, dim3(256), 0, stream, grp);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int TN, int TM, bool FAST>
static int launch_group_deq(GemmGroup<DequantParams> grp, hipStream_t stream) {
  const dim3 grid(group_tiles(&grp, 64 * TN, 64 * TM));
  launch_kernel((gemm_kblock_group_deq_kernel<TN, TM, FAST>), grid, dim3(256), 0, stream, grp);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

int launch_gemm_kblock_group(int tile, GemmGroup<RequantParams> grp, hipStream_t stream) {
  switch (tile) {
    case 44: return launch_group<4, 4>(grp, stream);
    case 34: return launch_group<3, 4>(grp, stream);
    case 22: return launch_group<2, 2>(grp, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

int launch_gemm_kblock_group(int tile, bool fast, GemmGroup<DequantParams> grp, hipStream_t stream) {
  switch (tile) {
    case 44: return fast ? launch_group_deq<4, 4, true>(grp, stream) : launch_group_deq<4, 4, false>(grp, stream);
    case 34: return fast ? launch_group_deq<3, 4, true>(grp, stream) : launch_group_deq<3, 4, false>(grp, stream);
    case 22: return fast ? launch_group_deq<2, 2, true>(grp, stream) : launch_group_deq<2, 2, false>(grp, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

}  // namespace mi
