// int8 GEMM with K split over the workgroups of a tile: shapes whose tiles leave CUs idle.
#include "gemm_ring.h"

namespace mi {

// =====================================================================================================================
// A tile's K blocks are dealt to `parts` workgroups.  Each leaves its int32 sums in memory, counts itself in, and is done, but for
// the last of them to arrive: that one adds the others' sums to its own and goes on as an unsplit tile would.  Nothing waits for
// another workgroup.  (int32 sums in any order are the same sums.)
// A CU gets 50 to 60 GB/s of operands where weights come from HBM (see gemm_ring.h), so what a launch takes is what its busiest CU
// has to fetch: split, more CUs share it, or larger tiles fetch less of it.  The sums cross the XCDs: they are written through and
// read past the L2s (agent scope), which makes the stores' completion all that has to be waited for before the count.
// =====================================================================================================================
constexpr int kAgentScope = 16;  // cache policy of an access at the device's coherence point (sc1)
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// bytes of a part's sums: 16 bytes per thread and quarter of an MFMA tile, behind them the row sums
template <int TN, int TM, bool HAS_ZW>
constexpr int part_bytes() { return 256 * (TN * TM * 64 + (HAS_ZW ? 16 : 0)); }

template <int TN, int TM, bool HAS_ZW>
__device__ __forceinline__ bool add_parts(const KPart &kp, v16i (&acc)[TN][TM], int (&rowsum)[TM], int *lds, int tid) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BYTES = part_bytes<TN, TM, HAS_ZW>(), V = TN * TM * 4, ALL = V + (HAS_ZW ? 1 : 0);
  static_assert(TM <= 4, "the row sums of a thread in 16 bytes");
  const __amdgpu_buffer_rsrc_t sums =
      __builtin_amdgcn_make_buffer_rsrc(kp.sums + (int64_t)kp.tile * kp.parts * BYTES, (short)0, kp.parts * BYTES, 0x00020000);
#pragma unroll
  for (int v = 0; v < ALL; ++v) {
    v4u x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (v < V) x[e] = (uint32_t)acc[v / 4 / TM % TN][v / 4 % TM][v % 4 * 4 + e];
      else x[e] = e < TM ? (uint32_t)rowsum[e % TM] : 0u;
    }
    __builtin_amdgcn_raw_buffer_store_b128(x, sums, (v * 256 + tid) * 16, kp.part * BYTES, kAgentScope);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's sums are where every CU reads them
  __syncthreads();
  if (tid == 0) *lds = (int)__hip_atomic_fetch_add(kp.arrived + kp.tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(*lds) != kp.parts - 1) return false;
  __syncthreads();  // (every wave has read the word; the LDS is the epilogue's from here on)
  if (tid == 0) __hip_atomic_store(kp.arrived + kp.tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  constexpr int AT_ONCE = TN * TM >= 4 ? 1 : 4 / (TN * TM);  // as many parts as fit 64 registers
  for (int p = 1; p < kp.parts; p += AT_ONCE) {              // counted from this workgroup's own
    v4u x[AT_ONCE][ALL];
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) {
      const int q = kp.part + (p + u < kp.parts ? p + u : 0), other = q < kp.parts ? q : q - kp.parts;  // (past the end: its own, unused)
#pragma unroll
      for (int v = 0; v < ALL; ++v)
        x[u][v] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(sums, (v * 256 + tid) * 16, other * BYTES, kAgentScope));
    }
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) {
      if (p + u < kp.parts) {
        // (every part started from kAccBias, which the epilogue takes out once)
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v16i &a = acc[v / 4 / TM][v / 4 % TM];
            a[v % 4 * 4 + e] = (int)((uint32_t)a[v % 4 * 4 + e] + x[u][v][e] - kAccBias);
          }
        if (HAS_ZW) {
#pragma unroll
          for (int j = 0; j < TM; ++j) rowsum[j] += (int)x[u][ALL - 1][j];
        }
      }
    }
  }
#endif
  return true;
}

template <int EPI>
struct SplitCall {
  GemmCall<EPI> call;
  int8_t *space;
  int parts;
};
static_assert(sizeof(SplitCall<EPI_REQUANT>) <= kShortArgs && sizeof(SplitCall<EPI_DEQUANT>) <= kShortArgs, "see launch_args.h");

template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST, bool STREAM>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(ring_occupancy<TN, TM, S>(), ring_occupancy<TN, TM, S>()))) void gemm_split_kernel(
        SplitCall<EPI> split) {
  GemmArgs g;
  RequantParams rq;
  DequantParams dq;
  split.call.open(&g, &rq, &dq);
  // part by part, so that the workgroups of an XCD read the same K range of the activations
  const int tiles = g.tiles_m * g.tiles_n, id = xcd_order((int)blockIdx.x, tiles * split.parts);
  KPart kp;
  kp.part = id / tiles;
  kp.parts = split.parts;
  kp.tile = id - kp.part * tiles;
  kp.arrived = reinterpret_cast<uint32_t *>(split.space);
  kp.sums = split.space + kSplitCounterBytes;
  int tile_m, tile_n;
  tile_of(g, kp.tile, &tile_m, &tile_n);
  gemm_ring_body<TN, TM, S, EPI, HAS_ZW, FAST, STREAM, true>(g, rq, dq, tile_m, tile_n, kp);
}

template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST>
static int launch(int parts, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, void *space, hipStream_t stream) {
  const SplitCall<EPI> split{GemmCall<EPI>::of(g, g.wb, 64 * TN, 64 * TM, rq, dq), static_cast<int8_t *>(space), parts};
  const int64_t tiles = (int64_t)split.call.tiles_m * split.call.tiles_n;
  if (parts < 2 || parts > (g.k + 127) / 128 || tiles * sizeof(uint32_t) > kSplitCounterBytes ||
      tiles * parts * part_bytes<TN, TM, HAS_ZW>() > (int64_t)kSplitSumBytes) {
    set_error("gemm: K in %d parts does not fit", parts);
    return MI_ERROR;
  }
  const dim3 grid((unsigned)(tiles * parts));
  if (split.call.tiles_m <= kStreamRowTiles) {
    launch_kernel((gemm_split_kernel<TN, TM, S, EPI, HAS_ZW, FAST, true>), grid, dim3(256), 0, stream, split);
  } else {
    launch_kernel((gemm_split_kernel<TN, TM, S, EPI, HAS_ZW, FAST, false>), grid, dim3(256), 0, stream, split);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int TN, int TM, int S>
static int with_form(int parts, bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                     void *space, hipStream_t stream) {
  if (requant && fast && has_zw) return launch<TN, TM, S, EPI_REQUANT, true, true>(parts, g, rq, dq, space, stream);
  if (requant && fast) return launch<TN, TM, S, EPI_REQUANT, false, true>(parts, g, rq, dq, space, stream);
  if (!requant && !has_zw && fast) return launch<TN, TM, S, EPI_DEQUANT, false, true>(parts, g, rq, dq, space, stream);
  if (!requant && !has_zw) return launch<TN, TM, S, EPI_DEQUANT, false, false>(parts, g, rq, dq, space, stream);
  set_error("gemm: no such form of a split K");
  return MI_ERROR;
}

thread_local SplitLaunches t_split_launches;

int launch_gemm_split(int tile, int parts, bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq,
                      const DequantParams &dq, void *space, hipStream_t stream) {
  if (g.wb == nullptr || space == nullptr) {
    set_error("gemm: the blocked weight copy or the space for split sums is missing");
    return MI_NULL_PTR;
  }
  t_split_launches = SplitLaunches{t_split_launches.count + 1, tile, parts};
  switch (tile) {
    case 11: return with_form<1, 1, 5>(parts, requant, has_zw, fast, g, rq, dq, space, stream);
    case 12: return with_form<1, 2, 6>(parts, requant, has_zw, fast, g, rq, dq, space, stream);
    case 22: return with_form<2, 2, 5>(parts, requant, has_zw, fast, g, rq, dq, space, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

}  // namespace mi
