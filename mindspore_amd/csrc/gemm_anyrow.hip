// int8 GEMM on the matrix cores for activation rows of any length at any address, on 64 x 64 tiles (gemm_i8.hip says which
// shapes come here).
#include "gemm_core.h"

namespace mi {

typedef v4i v4i_byte __attribute__((aligned(1)));

// =====================================================================================================================
// Activations through registers, four K blocks of 128 bytes at a time.
//
// The asynchronous loads into LDS of the other loops want rows of whole 16-byte chunks; a row length that is none costs a copy
// of the rows and a launch, and a small product takes little more than a launch itself.  A load into registers takes 16
// bytes from any address: here A goes that way, and into the places in LDS where the asynchronous loads would have put it.
// Bytes past K are cleared (row sums; the weights are zero there), and a chunk that would reach past the tensor is fetched
// from its last 16 bytes and shifted.  W comes as in gemm_ring.hip.
// LDS holds two sets of four blocks of both operands: one is computed on while the other arrives.  Four blocks, 64 KiB, are about
// what a CU can have on its way.
// Bound by launch and latency; per 512 bytes of K about 1 us, the time of 64 KiB per CU.  333 x 1001 x 1000 with weight zero
// points 8.3 us (copy and ring) -> 5.35; more figures and where it ends are at gemm_anyrow_takes.
// =====================================================================================================================
template <int EPI, bool HAS_ZW, bool FAST>
__device__ __forceinline__ void gemm_anyrow_body(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int TILE = 64, KB = 128, SET = 4, HALF = SET * TILE * KB;  // HALF: one operand's part of a set
  static_assert(4 * HALF >= kEpiArrays * TILE * 4 + epi_wg_bytes<EPI, 1, 1>(), "the epilogue staging must fit");
  __shared__ __attribute__((aligned(1024))) char lds[4 * HALF];

  int tile_m, tile_n;
  tile_coords(g, &tile_m, &tile_n);
  const int m0 = tile_m * TILE, n0 = tile_n * TILE;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  const int r = lane & 31, h = lane >> 5;
  const int last = (g.k + KB - 1) / KB - 1;
  EpiParams<TILE, EPI, FAST> epi;
  epi.fetch(rq, dq, n0, g.n, tid);
  DeqInput<1> din;
  if (EPI == EPI_DEQUANT) din.fetch_rows(dq, m0 + wm * 32, r, g.m);

  const int k64 = g.k_pad >> 6;
  const WaveWeightGroups<1> wg(g.n, n0, wave, kNPad);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t *>(g.wb) + (int64_t)wg.first * k64 * 1024, (short)0, wg.inside * k64 * 1024, 0x00020000);
  auto lds_ptr = [](char *p) { return (__attribute__((address_space(3))) void *)p; };
  // (past the last block: that block again, which nobody computes on)
  auto load_w = [&](int set) {
#pragma unroll
    for (int j = 0; j < SET; ++j) {
      const int kb = set * SET + j < last ? set * SET + j : last;
#pragma unroll
      for (int l = 0; l < 2; ++l)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, lds_ptr(lds + (set & 1) * 2 * HALF + j * TILE * KB + wave * 2048 + l * 1024), 16,
                                                 lane * 16, blocked_weight_offset(wg.group(0), l, k64, kb), 0, 0);
    }
  };

  // a wave fetches 16 rows, 8 per instruction, into the swizzled order of gemm_kblock_body
  const int drow = lane >> 3;
  const int8_t *a_chunk[2];
  int a_at[2];  // where in a block the chunk starts
  const int8_t *last16 = g.a + (int64_t)(g.m - 1) * g.lda + g.k - 16;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int m = m0 + wave * 16 + 8 * i + drow;
    m = m < g.m ? m : g.m - 1;
    a_at[i] = ((lane & 7) ^ (drow >> 1) ^ (i << 2)) << 4;
    a_chunk[i] = g.a + (int64_t)m * g.lda + a_at[i];
  }
  v4i x[SET][2];
  auto load_a = [&](int set) {
#pragma unroll
    for (int j = 0; j < SET; ++j) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int8_t *p = a_chunk[i] + (int64_t)(set * SET + j) * KB;
        x[j][i] = *reinterpret_cast<const v4i_byte *>(p < last16 ? p : last16);
      }
    }
  };
  auto store_a = [&](int set) {
#pragma unroll
    for (int j = 0; j < SET; ++j) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (set * SET + j == last) {
          const int64_t by = a_chunk[i] + (int64_t)last * KB - last16;
          const int have = g.k - last * KB - a_at[i];  // bytes of the chunk that exist
          unsigned __int128 v = __builtin_bit_cast(unsigned __int128, x[j][i]);
          if (by > 0) v = by < 16 ? v >> (8 * (int)by) : 0;
          if (have < 16) v = have > 0 ? v & (((unsigned __int128)1 << (8 * have)) - 1) : 0;
          x[j][i] = __builtin_bit_cast(v4i, v);
        }
        *reinterpret_cast<v4i *>(lds + ((set & 1) * 2 + 1) * HALF + j * TILE * KB + wave * 2048 + i * 1024 + lane * 16) = x[j][i];
      }
    }
  };

  v16i acc[1][1];
  int rowsum[1] = {0};
  const int w_off = (wn * 2 + (r >> 4)) * 2048 + h * 256 + (r & 15) * 16, a_off = HALF + (wm * 32 + r) * KB;
  const int swz = (r >> 1) & 7;
  auto compute = [&](const char *block) {
    v4i w[4], a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      w[q] = *reinterpret_cast<const v4i *>(block + w_off + (q >> 1) * 1024 + (q & 1) * 512);
      a[q] = *reinterpret_cast<const v4i *>(block + a_off + (((2 * q + h) ^ swz) << 4));
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (HAS_ZW) {
#pragma unroll
        for (int d = 0; d < 4; ++d) rowsum[0] = __builtin_amdgcn_sdot4(a[q][d], 0x01010101, rowsum[0], false);
      }
      acc[0][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[q], a[q], acc[0][0], 0, 0, 0);
    }
  };

  load_w(0);
  load_a(0);
  if (EPI == EPI_DEQUANT) din.fetch_tensor(dq);
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][0][e] = (int)kAccBias;
  store_a(0);
  const int sets = last / SET + 1;
  for (int set = 0; set < sets; ++set) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // this set is in, and the one before is done with
    if (set + 1 < sets) {
      load_w(set + 1);
      load_a(set + 1);
    }
    const char *mine = lds + (set & 1) * 2 * HALF;
#pragma unroll
    for (int j = 0; j < SET; ++j)
      if (set * SET + j <= last) compute(mine + j * TILE * KB);
    if (set + 1 < sets) store_a(set + 1);
  }
  __syncthreads();
  epi.to_lds(reinterpret_cast<int *>(lds), tid);
  gemm_epilogue<TILE, 1, 1, EPI, HAS_ZW, FAST, kAccBias, true>(
      acc, rowsum, g, rq, dq, din, reinterpret_cast<const int *>(lds), lds + kEpiArrays * TILE * 4 + wave * epi_stage_bytes<EPI, 1>(),
      lds + kEpiArrays * TILE * 4, n0, m0, n0 + wn * 32, m0 + wm * 32, r, h);
#endif
}

// (the LDS lets one workgroup into a CU: a wave per SIMD)
template <int EPI, bool HAS_ZW, bool FAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_anyrow_kernel(GemmCall<EPI> call) {
  GemmArgs g;
  RequantParams rq;
  DequantParams dq;
  call.open(&g, &rq, &dq);
  gemm_anyrow_body<EPI, HAS_ZW, FAST>(g, rq, dq);
}

template <int EPI, bool HAS_ZW, bool FAST>
static int launch(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  const auto call = GemmCall<EPI>::of(g, g.wb, 64, 64, rq, dq);
  launch_kernel((gemm_anyrow_kernel<EPI, HAS_ZW, FAST>), call.grid(), dim3(256), 0, stream, call);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

int launch_gemm_anyrow(bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                       hipStream_t stream) {
  if (!requant) {
    if (has_zw) return launch<EPI_DEQUANT, true, false>(g, rq, dq, stream);
    return launch<EPI_DEQUANT, false, false>(g, rq, dq, stream);
  }
  if (has_zw) return fast ? launch<EPI_REQUANT, true, true>(g, rq, dq, stream) : launch<EPI_REQUANT, true, false>(g, rq, dq, stream);
  return fast ? launch<EPI_REQUANT, false, true>(g, rq, dq, stream) : launch<EPI_REQUANT, false, false>(g, rq, dq, stream);
}

}  // namespace mi
