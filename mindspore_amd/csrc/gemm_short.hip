// int8 GEMM on the matrix cores, tiles of 32 rows whose K the waves of a workgroup share (gemm_i8.hip says which shapes come here).
#include "gemm_core.h"
#include "row_chunks.h"

namespace mi {

typedef v4i v4i_word __attribute__((aligned(4)));

// =====================================================================================================================
// Small products: many small tiles, and K shared out inside the workgroup.
//
// A product that one round of 64 x 64 tiles leaves most CUs out of lasts as long as one tile: launch, the way to the first operand, the K
// blocks one behind the other, requantisation and stores.  Here a tile is a quarter of that, so four times the CUs fetch, and its K blocks
// are dealt to 4 or 8 waves, each of which computes the whole tile over its own: no barrier until they meet once, in LDS, to add up (int32
// sums in any order are the same sums) and to requantise four channels of a row a lane.  The weights go from the blocked copy straight into
// operand registers, whole lines an instruction; the activations through an area of LDS that is the wave's own, since operand order from
// memory would look up 64 lines an instruction.
// Bound by launch and latency: 3.1 us is what a launch of one K block takes.  us per launch from a graph (K is not in parts there), ring -> this:
// 128 x 768 x 768 4.10 -> 3.42, 197 x 768 x 768 (fp32) 4.59 -> 3.52, 197 x 2304 x 768 (fp32) 4.79 -> 4.11, 197 x 768 x 3072 (fp32) 7.63 ->
// 4.78, 256 x 1024 x 1024 4.44 -> 3.73, 300 x 500 x 4096 8.74 -> 5.30; 64 rows, weights from HBM, decode kernel -> this: 4096 x 4096 8.8 ->
// 7.5, 1024 x 4096 7.9 -> 5.3.  Two K blocks a wave are on their way at a time; three or four gain nothing (128 x 768 x 768 3.47) and
// let fewer workgroups into a CU (197 x 3072 x 768 4.71 -> 5.86).
//
// ANY: rows of any length at any address.  Loads from odd addresses take the address unit about 95 cycles each, so what is fetched are the
// aligned 16-byte chunks that a row's bytes lie in, nine for 128 bytes, and the row comes into place on its way out of LDS: five dwords from
// the word it starts in and a byte shift (fragments read at odd addresses kept LDS busy for 14 cycles each, 3000 a CU at the first of the
// following).  A chunk may hold up to 15 bytes in front of the tensor or behind it: in memory they share its 16 bytes and so its page, in
// the products they meet zero weights (or lie in front of the row), and the row sums leave them out.  333 x 1001 x 1000 with weight zero
// points 5.6 (gemm_anyrow.hip) -> 4.9 (odd reads) -> 4.75, 200 x 1000 x 1501 6.3 -> 4.84 -> 4.46, 90 x 700 x 3001 - -> 5.9 -> 5.1, 70 x 64 x 1003
// 5.81 -> 4.00 -> 3.75, 100 x 500 x 501 4.27 -> 3.50 -> 3.33.
// =====================================================================================================================
template <int WAVES, int TN, int EPI, bool HAS_ZW, bool ANY>
__device__ __forceinline__ void gemm_short_body(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int D = 2, KB = 128, PITCH = ANY ? KB + 16 : KB, LOADS = ANY ? 5 : 4, SLOT = LOADS * 1024, PIECES = 4 * TN, SUMS = PIECES * 1024 + (HAS_ZW ? 256 : 0);
  constexpr int AREA = D * SLOT > SUMS ? D * SLOT : SUMS;  // a wave's own LDS: its activations, then its sums
  __shared__ __attribute__((aligned(1024))) char lds[WAVES * AREA];

  int tile_m, tile_n;
  tile_coords(g, &tile_m, &tile_n);
  const int m0 = tile_m * 32, n0 = tile_n * 32 * TN;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int blocks = (g.k + KB - 1) / KB, first = wave * blocks / WAVES, end = (wave + 1) * blocks / WAVES;
  char *const mine = lds + wave * AREA;

  // weights straight into operand registers: a fragment is two pieces of 512 bytes of the blocked copy
  const int k64 = g.k_pad >> 6;
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t *>(g.wb) + (int64_t)(n0 >> 4) * k64 * 1024, (short)0, 2 * TN * k64 * 1024, 0x00020000);
  const int w_at = (r >> 4) * k64 * 1024 + h * 256 + (r & 15) * 16;
  v4i w[D][4][TN];
  auto load_w = [&](int s, int kb) {
#pragma unroll
    for (int f = 0; f < 4; ++f) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
        w[s][f][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_at + i * 2 * k64 * 1024, kb * 2048 + f * 512, 0));
    }
  };

  // Activations through LDS, 16 bytes a lane, front to back.  Whole chunks: 8 rows x 128 bytes an instruction, chunks swizzled as in
  // gemm_kblock_body.  Any rows: the nine aligned chunks that a row's 128 bytes lie in.
  const int last = blocks - 1;
  const int8_t *const a_tile = g.a + (int64_t)m0 * g.lda;
  const int rows = min(g.m - m0, 32);
  const RowChunks ragged(reinterpret_cast<uintptr_t>(a_tile), g.m - m0, g.k);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(a_tile) - (ANY ? ragged.skew : 0), (short)0, -1, 0x00020000);
  int a_off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    a_off[i] = ANY ? ragged.first(i * 64 + lane)
                   : min(8 * i + (lane >> 3), rows - 1) * (int)g.lda + (((lane & 7) ^ (lane >> 4) ^ ((i & 1) << 2)) << 4);
  auto load_a = [&](int s, int kb) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int off = ANY ? ragged.of_block(a_off[i], kb) : a_off[i] + kb * KB;
      if (!ANY && kb == last) {  // (a chunk past K: the row's last one again)
        const int at = ((lane & 7) ^ (lane >> 4) ^ ((i & 1) << 2)) << 4;
        off += min(g.k - 16 - last * KB - at, 0);
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (__attribute__((address_space(3))) void *)(mine + s * SLOT + i * 1024), 16, off, 0, 0, 0);
    }
  };

  // the pieces that this wave finishes: four channels of a row a lane
  constexpr int OWN = PIECES / WAVES > 0 ? PIECES / WAVES : 1;
  int channel[OWN];
#pragma unroll
  for (int t = 0; t < OWN; ++t) {
    const int piece = wave * OWN + t;
    channel[t] = n0 + 8 * (piece < PIECES ? piece : 0) + 4 * h;
  }
  v4i par[OWN][6];
  auto load_params = [&] {
#pragma unroll
    for (int t = 0; t < OWN; ++t) {
      auto four = [&](const auto *p) { return *reinterpret_cast<const v4i *>(p + channel[t]); };
      if constexpr (EPI == EPI_REQUANT) {
        par[t][0] = four(rq.mult2);
        par[t][1] = four(rq.c2lo);
        par[t][2] = four(rq.c2hi);
        par[t][3] = four(rq.pre);
        par[t][4] = four(rq.rshift);
        if (HAS_ZW) par[t][5] = four(rq.zw);
      } else {
        par[t][0] = four(dq.wscale);
        par[t][1] = four(dq.wsum);
        par[t][2] = four(dq.bias);
      }
    }
  };
  DeqInput<1> din;

  v16i acc[TN];
  RowSums<1> sums;
  if (HAS_ZW) sums.clear(lane);
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = wave == 0 ? (int)kAccBias : 0;
  const uint32_t odd = ANY ? ragged.odd(r) : 0;
  const char *const row = mine + r * PITCH + (odd & ~3u);
  for (int b = first; b == first || b < end; b += D) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      if (b + s < end) {
        load_a(s, b + s);
        load_w(s, b + s);
      }
    }
    if (b == first) {
      load_params();
      if (EPI == EPI_DEQUANT) {
        din.fetch_rows(dq, m0, r, g.m);
        din.fetch_tensor(dq);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int s = 0; s < D; ++s) {
      if (b + s < end) {
        v4i a[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          if constexpr (ANY) {
            const char *at = row + s * SLOT + 32 * f + 16 * h;
            const v4i v = *reinterpret_cast<const v4i_word *>(at);
            const uint32_t next = *reinterpret_cast<const uint32_t *>(at + 16);
#pragma unroll
            for (int d = 0; d < 4; ++d) a[f][d] = (int)__builtin_amdgcn_alignbyte(d < 3 ? (uint32_t)v[(d + 1) & 3] : next, (uint32_t)v[d], odd & 3);
          } else {
            a[f] = *reinterpret_cast<const v4i *>(row + s * SLOT + (((2 * f + h) ^ ((r >> 1) & 7)) << 4));
          }
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          if (HAS_ZW) {
            v4i one[1] = {a[f]};
            if (b + s == last) {  // bytes past K are no part of the row
              int have = 8 * (g.k - last * KB - 32 * f - 16 * h);
              asm volatile("" : "+v"(have));  // (here, and not for every place at once before the loop)
#pragma unroll
              for (int d = 0; d < 4; ++d) one[0][d] &= (int)(((uint64_t)1 << max(min(have - 32 * d, 32), 0)) - 1);
            }
            sums.add(one, true);
          }
#pragma unroll
          for (int i = 0; i < TN; ++i) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[s][f][i], a[f], acc[i], 0, 0, 0);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every fragment is read before its place is filled again
  }

#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<v4i *>(mine + (4 * i + q) * 1024 + lane * 16) = v4i{acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
  if (HAS_ZW) {
    int rowsum[1];
    sums.get(rowsum);
    *reinterpret_cast<int *>(mine + PIECES * 1024 + lane * 4) = rowsum[0];
  }
  __syncthreads();
  if (wave * OWN >= PIECES) return;
  uint32_t rowsum = 0;
  if (HAS_ZW) {
#pragma unroll
    for (int o = 0; o < WAVES; ++o) rowsum += *reinterpret_cast<const uint32_t *>(lds + o * AREA + PIECES * 1024 + lane * 4);
    rowsum += (uint32_t)__shfl_xor((int)rowsum, 32);
  }
  const int m = m0 + r;
#pragma unroll
  for (int t = 0; t < OWN; ++t) {
    uint32_t v[4] = {};
#pragma unroll
    for (int o = 0; o < WAVES; ++o) {
      const v4i part = *reinterpret_cast<const v4i *>(lds + o * AREA + (wave * OWN + t) * 1024 + lane * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += (uint32_t)part[e];
    }
    const int n = channel[t];
    if constexpr (EPI == EPI_REQUANT) {
      // as in gemm_epilogue
      int y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (HAS_ZW) v[e] -= rowsum * (uint32_t)par[t][5][e];
        const uint64_t c2 = ((uint64_t)(uint32_t)par[t][2][e] << 32) | (uint32_t)par[t][1][e];
        uint64_t p2, carry, unused;
        int32_t x;
        asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=&v"(p2), "=s"(carry) : "v"(v[e]), "v"(par[t][0][e]), "v"(c2));
        asm("v_addc_co_u32_e64 %0, %1, %2, %3, %4" : "=v"(x), "=s"(unused) : "v"((int32_t)(p2 >> 32)), "v"(par[t][3][e]), "s"(carry));
        y[e] = med3_i32(x >> par[t][4][e], rq.amin, rq.amax);
      }
      const uint32_t four = pack4(y[0], y[1], y[2], y[3]);
      int8_t *c = static_cast<int8_t *>(g.c) + (int64_t)m * g.ldc + n;
      if (m < g.m) {
        if (n + 4 <= g.n) {
          *reinterpret_cast<u32_any *>(c) = four;
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (n + e < g.n) c[e] = (int8_t)(four >> (8 * e));
        }
      }
    } else {
      const bool with_act = dq.act == MI_ACT_RELU || dq.act == MI_ACT_RELU6;
      const float act_lo = with_act ? 0.0f : -__builtin_inff();
      const float act_hi = dq.act == MI_ACT_RELU6 ? 6.0f : __builtin_inff();
      const uint32_t kzz = (uint32_t)dq.deep * (uint32_t)din.zx * (uint32_t)dq.zw0;
      v4f o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t u = v[e] + kzz - (uint32_t)din.zx * (uint32_t)par[t][1][e] - kAccBias;
        if (HAS_ZW) u -= (uint32_t)dq.zw0 * rowsum;
        float d = __fmul_rn(__fmul_rn(din.sxr[0], __int_as_float(par[t][0][e])), (float)(int32_t)u);
        if (dq.has_bias) d = __fadd_rn(d, __int_as_float(par[t][2][e]));
        d = (act_lo > d) ? act_lo : d;
        o[e] = (act_hi < d) ? act_hi : d;
      }
      float *c = static_cast<float *>(g.c) + (int64_t)m * g.ldc + n;
      if (m < g.m) {
        if (n + 4 <= g.n) {
          *reinterpret_cast<v4f_any *>(c) = o;
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (n + e < g.n) c[e] = o[e];
        }
      }
    }
  }
#endif
}

template <int WAVES, int TN, int EPI, bool HAS_ZW, bool ANY>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2))) void gemm_short_kernel(GemmCall<EPI> call) {
  GemmArgs g;
  RequantParams rq;
  DequantParams dq;
  call.open(&g, &rq, &dq);
  gemm_short_body<WAVES, TN, EPI, HAS_ZW, ANY>(g, rq, dq);
}

template <int WAVES, int TN, bool ANY, int EPI, bool HAS_ZW>
static int launch(const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  const auto call = GemmCall<EPI>::of(g, g.wb, 32 * TN, 32, rq, dq);
  launch_kernel((gemm_short_kernel<WAVES, TN, EPI, HAS_ZW, ANY>), call.grid(), dim3(64 * WAVES), 0, stream, call);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int WAVES, int TN, bool ANY>
static int with_form(bool requant, bool has_zw, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq, hipStream_t stream) {
  if (requant && has_zw) return launch<WAVES, TN, ANY, EPI_REQUANT, true>(g, rq, dq, stream);
  if (requant) return launch<WAVES, TN, ANY, EPI_REQUANT, false>(g, rq, dq, stream);
  if (has_zw) return launch<WAVES, TN, ANY, EPI_DEQUANT, true>(g, rq, dq, stream);
  return launch<WAVES, TN, ANY, EPI_DEQUANT, false>(g, rq, dq, stream);
}

template <bool ANY>
static int with_tile(int tile, bool requant, bool has_zw, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                     hipStream_t stream) {
  switch (tile) {
    case 41: return with_form<4, 1, ANY>(requant, has_zw, g, rq, dq, stream);
    case 81: return with_form<8, 1, ANY>(requant, has_zw, g, rq, dq, stream);
    case 82: return with_form<8, 2, ANY>(requant, has_zw, g, rq, dq, stream);
  }
  set_error("gemm: no such tile (%d)", tile);
  return MI_ERROR;
}

int launch_gemm_short(int tile, bool any, bool requant, bool has_zw, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                      hipStream_t stream) {
  if (g.wb == nullptr) {
    set_error("gemm: the blocked weight copy is missing");
    return MI_NULL_PTR;
  }
  if (any && g.lda != g.k) {  // (RowChunks)
    set_error("gemm: rows of %d bytes %lld apart", g.k, (long long)g.lda);
    return MI_PARAM_INVALID;
  }
  return any ? with_tile<true>(tile, requant, has_zw, g, rq, dq, stream) : with_tile<false>(tile, requant, has_zw, g, rq, dq, stream);
}

}  // namespace mi
