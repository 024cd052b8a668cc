// int8 GEMM on the matrix cores, K in blocks of 128 bytes through a ring of LDS stages (gemm_i8.hip says which shapes come
// here).
#include "gemm_ring.h"

namespace mi {

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

template <int TN, int TM, int S, int EPI, bool HAS_ZW, bool FAST>
static int launch_ring(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  const auto call = GemmCall<EPI>::of(g, g.wb, 64 * TN, 64 * TM, rq, dq);
  if (call.tiles_m <= kStreamRowTiles) {
    launch_kernel((gemm_ring_kernel<TN, TM, S, EPI, HAS_ZW, FAST, true>), call.grid(), dim3(256), 0, stream, call);
  } else {
    launch_kernel((gemm_ring_kernel<TN, TM, S, EPI, HAS_ZW, FAST, false>), call.grid(), dim3(256), 0, stream, call);
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
    launch_kernel((gemm_ring_group_kernel<TN, TM, S, true>), grid, dim3(256), 0, stream, grp);
  } else {
    launch_kernel((gemm_ring_group_kernel<TN, TM, S, false>), grid, dim3(256), 0, stream, grp);
  }
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int TN, int TM, int S, bool FAST>
static int launch_group_deq(GemmGroup<DequantParams> grp, hipStream_t stream) {
  const dim3 grid(group_tiles(&grp, 64 * TN, 64 * TM));
  if (grp.g.tiles_m <= kStreamRowTiles) {
    launch_kernel((gemm_ring_group_deq_kernel<TN, TM, S, FAST, true>), grid, dim3(256), 0, stream, grp);
  } else {
    launch_kernel((gemm_ring_group_deq_kernel<TN, TM, S, FAST, false>), grid, dim3(256), 0, stream, grp);
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
