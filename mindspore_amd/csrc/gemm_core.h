// What the int8 GEMM kernels of all main loops share: arguments, tile order, fused epilogues, operand fragments.
#pragma once

#include "common.h"
#include "launch_args.h"
#include "quant_math.h"
#include "weight_loads.h"

#include <type_traits>

namespace mi {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
// the same at any address: C rows start wherever the caller's row length puts them, and the hardware stores 4 or 16 bytes
// to any byte address in one instruction
typedef v4i v4i_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef v4f v4f_any __attribute__((aligned(4)));

enum { EPI_REQUANT = 0, EPI_DEQUANT = 1 };

struct GemmArgs {
  const int8_t *a;
  int64_t lda;
  int m;
  int k;  // bytes of K that may be read from A (multiple of 16)
  const int8_t *w;
  int ldw;    // weight row stride in bytes
  int k_pad;  // contraction extent of the packed weights (zero filled past K)
  const int8_t *wb;  // the blocked copy of the weights (WeightView::blocked) or nullptr
  int n;
  int tiles_m, tiles_n;
  void *c;
  int64_t ldc;
  uint32_t group_magic;  // quotients by 4 * tiles_n (see magic31)
  int group_shift;
};

// The arguments of one matrix as they travel; w: the form of the weights that the kernel reads, c: rows of n values.
template <int EPI>
struct GemmCall {
  typedef std::conditional_t<EPI == EPI_REQUANT, RequantCall, DequantCall> Epi;
  const int8_t *a, *w;
  void *c;
  int m, n, k, lda, tiles_m, tiles_n;
  uint32_t group_magic;
  int group_shift;
  Epi epi;
  static GemmCall of(const GemmArgs &g, const int8_t *w, int tile_n, int tile_m, const RequantParams &rq, const DequantParams &dq) {
    GemmCall call{g.a, w, g.c, g.m, g.n, g.k, (int)g.lda, (g.m + tile_m - 1) / tile_m, (g.n + tile_n - 1) / tile_n, 0, 0, {}};
    magic31(4 * call.tiles_n, &call.group_magic, &call.group_shift);
    if constexpr (EPI == EPI_REQUANT) call.epi = RequantCall::of(rq);
    else call.epi = DequantCall::of(dq, g.k);
    return call;
  }
  dim3 grid() const { return dim3(tiles_m * tiles_n); }
  __device__ __forceinline__ void open(GemmArgs *g, RequantParams *rq, DequantParams *dq) const {
    // all arguments in one go: left to itself the compiler loads some where they are used, one way to memory behind the other
    asm volatile("" ::"s"(a), "s"(w), "s"(c), "s"(m), "s"(n), "s"(k), "s"(lda), "s"(tiles_m), "s"(tiles_n), "s"(group_magic),
                 "s"(group_shift), "s"(epi.channels));
    const int k_pad = padded_k(k);
    *g = GemmArgs{a, lda, m, k, w, weight_row_stride(k_pad), k_pad, w, n, tiles_m, tiles_n, c, n, group_magic, group_shift};
    if constexpr (EPI == EPI_REQUANT) {
      asm volatile("" ::"s"(epi.zo), "s"(epi.amin), "s"(epi.amax), "s"(epi.forms));
      *rq = epi.open(n);
    } else {
      asm volatile("" ::"s"(epi.qp_dev), "s"(epi.sx), "s"(epi.zx), "s"(epi.zw0), "s"(epi.forms));
      *dq = epi.open(n, k);
    }
  }
};
static_assert(sizeof(GemmCall<EPI_REQUANT>) <= kShortArgs && sizeof(GemmCall<EPI_DEQUANT>) <= kShortArgs, "see launch_args.h");

// Asynchronous 16-byte-per-lane copy global -> LDS: lane L's 16 bytes land at lds_wave_base + 16 * L;
// lds_wave_base must be wave-uniform.  Completion is tracked by vmcnt, in issue order.
__device__ __forceinline__ void async_copy16(const void *global_src, void *lds_wave_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)global_src,
                                   (__attribute__((address_space(3))) void *)lds_wave_base, 16, 0, 0);
}

// Hardware deals consecutive workgroup ids round-robin over the 8 XCDs (each with its own L2), so ids that share an
// XCD are mapped to a compact block of tiles, 4 tiles tall: the CUs of one XCD then share operand panels in L2.
__device__ __forceinline__ int xcd_order(int id, int grid) {
  const int per = grid >> 3;
  return id < per * 8 ? (id & 7) * per + (id >> 3) : id;
}
template <bool MAGIC = true>  // false: g has no group_magic
__device__ __forceinline__ void tile_of(const GemmArgs &g, int id, int *tile_m, int *tile_n) {
  constexpr int G = 4;
  const int width = G * g.tiles_n;
  const int group = MAGIC ? quotient31(id, g.group_magic, g.group_shift) : id / width, first = group * G;
  const int gsize = min(g.tiles_m - first, G), rest = id - group * width;
  // (rest < 2^29, so that its third, by a factor just above 2^32 / 3, is exact)
  *tile_n = gsize == 4 ? rest >> 2 : gsize == 3 ? (int)__umulhi((uint32_t)rest, 0x55555556u) : gsize == 2 ? rest >> 1 : rest;
  *tile_m = first + rest - *tile_n * gsize;
}
template <bool MAGIC = true>
__device__ __forceinline__ void tile_coords(const GemmArgs &g, int *tile_m, int *tile_n) {
  tile_of<MAGIC>(g, xcd_order((int)blockIdx.x, g.tiles_m * g.tiles_n), tile_m, tile_n);
}

// Several weight matrices with the same K against the same activation rows as one launch: their column tiles stand side by
// side, and a workgroup first finds the member its tile belongs to.  Fields are picked with selects over constant indices (a
// dynamically indexed kernel argument would be copied to scratch memory).
constexpr int kGemmGroupMax = 4;
template <typename P>  // P: the members' epilogue parameters (RequantParams or DequantParams)
struct GemmGroup {
  GemmArgs g;  // what they share; tiles_n counts the column tiles of all of them
  int count;
  int first_tile[kGemmGroupMax];  // a member's first column tile
  int n[kGemmGroupMax];
  const int8_t *wb[kGemmGroupMax];
  void *c[kGemmGroupMax];  // rows of n values
  P p[kGemmGroupMax];
};

template <typename P>
__device__ __forceinline__ void pick_member(const GemmGroup<P> &grp, int *tile_n, GemmArgs *g, P *p) {
  int first = 0;
  *g = grp.g;
  *p = grp.p[0];
  g->wb = grp.wb[0];
  g->n = grp.n[0];
  g->c = grp.c[0];
#pragma unroll
  for (int i = 1; i < kGemmGroupMax; ++i) {
    if (i < grp.count && *tile_n >= grp.first_tile[i]) {
      *p = grp.p[i];
      g->wb = grp.wb[i];
      g->n = grp.n[i];
      g->c = grp.c[i];
      first = grp.first_tile[i];
    }
  }
  g->ldc = g->n;
  *tile_n -= first;
}

// Host side: the grid of a group on tiles of tile_n channels x tile_m rows.
template <typename P>
int group_tiles(GemmGroup<P> *grp, int tile_n, int tile_m) {
  grp->g.tiles_m = (grp->g.m + tile_m - 1) / tile_m;
  grp->g.tiles_n = 0;
  for (int i = 0; i < grp->count; ++i) {
    grp->first_tile[i] = grp->g.tiles_n;
    grp->g.tiles_n += (grp->n[i] + tile_n - 1) / tile_n;
  }
  magic31(4 * grp->g.tiles_n, &grp->g.group_magic, &grp->g.group_shift);
  return grp->g.tiles_m * grp->g.tiles_n;
}

// clamp to [lo, hi] in one instruction (valid for lo <= hi)
__device__ __forceinline__ int med3_i32(int x, int lo, int hi) {
  int y;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(y) : "v"(x), "v"(lo), "v"(hi));
  return y;
}

__device__ __forceinline__ uint32_t pack4(int y0, int y1, int y2, int y3) {
  // low bytes of four ints -> one dword (v_perm_b32 x3)
  const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)y1, (uint32_t)y0, 0x0c0c0400u);
  const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)y3, (uint32_t)y2, 0x0c0c0400u);
  return __builtin_amdgcn_perm(p23, p01, 0x05040100u);
}

// ---- epilogue.  acc[i][j][4*q + e] is output channel n_w + 32*i + 8*q + 4*h + e of output row m_w + 32*j + r.
//      C rows are written with 4- and 16-byte stores at whatever alignment n and ldc leave them (a padded scratch output
//      and a pass that compacts it cost 333 x 1001 outputs 2.7 us, and 1-byte accesses at any size); the up to three
//      columns of the last, partial group of four go out one by one. ----
//      Per-channel parameters are read from LDS (array p of kEpiArrays x TILE_N ints, filled by EpiParams below):
//      global loads here would share the vmcnt counter with the output stores and serialise on them. ----
constexpr int kEpiArrays = 6;
constexpr int kDeqStageRowBytes = 144;  // fp32 output staging: 32 columns (128 B) + 16 B so that rows shift banks
// bytes of the wave-private output staging tile behind the parameter arrays
template <int EPI, int TM>
constexpr int epi_stage_bytes() { return EPI == EPI_REQUANT ? 16384 : TM * 32 * kDeqStageRowBytes; }
// row stride of the int8 staging tile that a workgroup of any other shape than 2 x 2 or 4 x 4 shares (16 bytes of
// padding: rows shift banks and stay 16-byte aligned)
template <int TN>
constexpr int epi_row_bytes() { return 64 * TN + 16; }
// all of a workgroup's staging
template <int EPI, int TN, int TM>
constexpr int epi_wg_bytes() {
  return EPI == EPI_DEQUANT     ? 4 * epi_stage_bytes<EPI, TM>()
         : TN == 4 && TM == 4   ? 4 * 16384
         : TN == 2 && TM == 2   ? 16384
                                : 64 * TM * epi_row_bytes<TN>();
}

// The workgroup's per-channel epilogue parameters: thread t holds channel n0 + t of each array (fetched at kernel
// start, so the latency is hidden by the main loop) and drops them into LDS once the main loop is done.
template <int TILE_N, int EPI, bool FAST>
struct EpiParams {
  int v[kEpiArrays];
  __device__ __forceinline__ void fetch(const RequantParams &rq, const DequantParams &dq, int n0, int n_total, int tid) {
#pragma unroll
    for (int a = 0; a < kEpiArrays; ++a) v[a] = 0;
    if (tid < TILE_N) {
      int n = n0 + tid;  // arrays are padded to a multiple of 256 channels, past which a tile of 192 can reach
      if (kNPad % TILE_N != 0) n = n < n_total ? n : n_total - 1;
      if (EPI == EPI_REQUANT && FAST) {
        v[0] = (int)rq.mult2[n];
        v[1] = (int)rq.c2lo[n];  // arrays 1 and 2 are interleaved in LDS: {lo, hi} of channel t at 2 * t
        v[2] = (int)rq.c2hi[n];
        v[3] = rq.pre[n];
        v[4] = rq.rshift[n];
        v[5] = rq.zw[n];
      } else if (EPI == EPI_REQUANT) {
        const RequantChannel ch = rq.each[n];
        v[0] = ch.mult;
        v[1] = ch.bias2;
        v[2] = ch.rshift();
        v[3] = ch.zw;
        v[4] = ch.lshift();
      } else {
        v[0] = __float_as_int(dq.wscale[n]);
        v[1] = dq.wsum[n];
        v[2] = __float_as_int(dq.bias[n]);
      }
    }
  }
  // call after a barrier that follows the last LDS read of the main loop; ends with a barrier
  __device__ __forceinline__ void to_lds(int *p, int tid) const {
    if (tid < TILE_N) {
#pragma unroll
      for (int a = 0; a < kEpiArrays; ++a) {
        if (EPI == EPI_REQUANT && FAST && (a == 1 || a == 2)) {
          p[TILE_N + 2 * tid + (a - 1)] = v[a];
        } else {
          p[a * TILE_N + tid] = v[a];
        }
      }
    }
    __syncthreads();
  }
};

// What the fp32 epilogue needs of the input's quantisation.  With DynamicQuant upstream the values live in device
// memory; they are fetched before the main loop, which hides a dependent load of a microsecond that would otherwise
// sit between the last MFMA and the first store of every tile.  The rows' scales are vector loads, which the main loops want ahead of
// their own; the tensor's come by scalar loads, and every scalar wait is for all of them: asked for before the first operand loads,
// they held those up by their whole way to memory.
template <int TM>
struct DeqInput {
  float sx;
  int32_t zx;
  float sxr[TM];  // per_row: the scale of the rows this lane holds
  __device__ __forceinline__ void fetch_rows(const DequantParams &dq, int m_w, int r, int m_total) {
    // input_per_channel_: one input scale per row (NN/int8/dynamic_matmul_int8.c:126-128)
    if (!dq.per_row) return;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      int m = m_w + j * 32 + r;
      m = m < m_total ? m : m_total - 1;
      sxr[j] = dq.qp_dev[m].scale_f;
    }
  }
  __device__ __forceinline__ void fetch_tensor(const DequantParams &dq) {  // behind the first operand loads
    asm volatile("" ::: "memory");
    sx = dq.sx;
    zx = dq.zx;
    if (dq.qp_dev != nullptr) {
      sx = dq.qp_dev->scale_f;
      zx = dq.qp_dev->zero_point;
    }
    if (!dq.per_row) {
#pragma unroll
      for (int j = 0; j < TM; ++j) sxr[j] = sx;
    }
  }
};

// ACC0: the value the accumulators started from (see kAccBias); it leaves through the per-channel constants, so it
// costs nothing here.
// STAGE: the LDS has room for the workgroup's whole int8 tile (epi_wg_bytes); without it, tiles other than 2 x 2 and 4 x 4
// are stored straight from the accumulator layout.
template <int TILE_N, int TN, int TM, int EPI, bool HAS_ZW, bool FAST, uint32_t ACC0 = 0, bool STAGE = false>
__device__ __forceinline__ void gemm_epilogue(v16i (&acc)[TN][TM], int (&rowsum)[TM], const GemmArgs &g,
                                              const RequantParams &rq, const DequantParams &dq,
                                              const DeqInput<TM> din, const int *p, char *cstage, char *cstage_wg,
                                              int n_tile, int m_tile, int n_w, int m_w, int r, int h) {
  static_assert(!(EPI == EPI_REQUANT && FAST) || ACC0 == kAccBias, "the host folds kAccBias into c2");
  if (HAS_ZW) {
#pragma unroll
    for (int j = 0; j < TM; ++j) rowsum[j] += __shfl_xor(rowsum[j], 32);
  }
  if (EPI == EPI_REQUANT) {
    int8_t *c = static_cast<int8_t *>(g.c);
    int amin_v = rq.amin, amax_v = rq.amax;
    asm volatile("" : "+v"(amin_v), "+v"(amax_v));  // kept in vector registers, as v_med3 wants them
    // A 128-channel-wide wave tile goes through LDS so that global memory sees whole 128-byte rows: written
    // straight from the accumulator layout, every store instruction would touch 32 rows with 8 bytes each, and the
    // L2 write path then becomes the bottleneck of the whole kernel.  Wave-private staging tile, 128 rows x 128 B:
    // 16-byte chunk c of row R sits at slot c ^ (R & 7), and inside a chunk dword d sits at (d + (R >> 3)) & 3, which
    // makes both the dword writes (32 rows, one column) and the 16-byte row reads bank-conflict free.
    // The output leaves at memory-write speed (all workgroups reach this point together), and a store instruction
    // that finds the write queue full holds up the wave: so the tile is requantised in two halves of 64 rows, and the
    // eight store instructions of the first half are issued one at a time between the pieces of the second.  (Four
    // passes of 32 rows would hide more of the stores, but every pass re-reads the per-channel constants from LDS,
    // and at four passes those reads take longer than the arithmetic.)
    constexpr bool kStageC = (TN == 4 && TM == 4);
    // The 128 x 128 tile (four wave tiles of 64 channels x 64 rows) does the same through ONE staging tile of
    // 128 rows x 128 B shared by the workgroup (same layout), so that its rows, too, leave as whole 128-byte lines:
    // every wave drops its quadrant, the workgroup meets, every wave stores 32 rows.  Straight from the accumulator
    // layout the stores were a quarter to a third of the launch time of mid-sized shapes (4096 x 1024 x 1024: 2.3 of
    // 9.0 us, 3136 x 2048 x 512: 3.3 of 10.0 us).
    constexpr bool kStageWG = (TN == 2 && TM == 2);
    // Tiles of other shapes in the K-block loop: one staging tile of the whole workgroup, rows of 64 TN + 16 bytes.
    constexpr bool kStageAny = STAGE && !kStageC && !kStageWG;
    const int wn_id = (n_w - n_tile) / (32 * TN), wm_id = (m_w - m_tile) / (32 * TM);
    const int lane = h * 32 + r;
    // four outputs (consecutive channels of one row): accumulator registers -> clamped int32
    auto requant4 = [&](const int32_t (&accv)[4], int rsum, v4i mult, v4i c2lo, v4i c2hi, v4i pre, v4i bias, v4i e4,
                        v4i ls, v4i zw, int (&y)[4]) {
      if (FAST) {
        // the host proved that the accumulator register, read as unsigned, stays below 2^31, that c2 is negative and
        // that none of the sums below leaves its type (RequantParams::fast2).  p2 = a * mult2 + c2 as unsigned 64-bit
        // numbers carries out exactly when the true (signed) sum is >= 0, i.e. when x >= 0: the carry is the
        // "+1 unless negative" of the rounding, so pre arrives here as pre - 1.  The four chains are written stage
        // by stage so that no instruction waits for the one before it.
        uint64_t p2[4], carry[4], unused;
        int32_t t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t a = (uint32_t)accv[e];
          if (HAS_ZW) a -= (uint32_t)rsum * (uint32_t)zw[e];
          const uint64_t c2 = ((uint64_t)(uint32_t)c2hi[e] << 32) | (uint32_t)c2lo[e];
          asm("v_mad_u64_u32 %0, %1, %2, %3, %4" : "=&v"(p2[e]), "=s"(carry[e]) : "v"(a), "v"(mult[e]), "v"(c2));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          asm("v_addc_co_u32_e64 %0, %1, %2, %3, %4"
              : "=v"(t[e]), "=s"(unused)
              : "v"((int32_t)(p2[e] >> 32)), "v"(pre[e]), "s"(carry[e]));
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] >>= e4[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = med3_i32(t[e], amin_v, amax_v);
        return;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t v = (uint32_t)accv[e];
        if (HAS_ZW) v -= (uint32_t)rsum * (uint32_t)zw[e];
        v += (uint32_t)bias[e];
        int32_t t = rdiv_pot(srdhm((int32_t)(v << ls[e]), mult[e]), e4[e]);
        t = (int32_t)((uint32_t)t + (uint32_t)rq.zo);
        t = t < rq.amax ? t : rq.amax;
        y[e] = t > rq.amin ? t : rq.amin;
      }
    };
    // The body is compiled twice: for wave tiles that lie wholly inside the matrix (no bounds checks, no divergent
    // branches around the stores) and for the ragged rest.
    const bool full_tile = kStageWG || kStageAny ? m_tile + 64 * TM <= g.m && n_tile + 64 * TN <= g.n
                                    : m_w + 32 * TM <= g.m && n_w + 32 * TN <= g.n;
    auto store4 = [&](int8_t *dst, int n, uint32_t four) {  // columns n .. n + 3 of a row, as far as they exist
      if (n + 4 <= g.n) {
        *reinterpret_cast<u32_any *>(dst) = four;
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (n + e < g.n) dst[e] = (int8_t)(four >> (8 * e));
      }
    };
    auto store16 = [&](int8_t *dst, int n, v4i o) {
      if (n + 16 <= g.n) {
        *reinterpret_cast<v4i_any *>(dst) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) store4(dst + 4 * e, n + 4 * e, (uint32_t)o[e]);
      }
    };
    auto body = [&](auto full_c) {
      constexpr bool FULL = decltype(full_c)::value;
      // rows lrow + 8 * t of the staging tile -> global memory (t: 0..15, one store instruction)
      auto store_rows = [&](int t) {
        const int c16 = lane & 7, lrow = lane >> 3;
        const int n = n_w + c16 * 16;
        const int row = lrow + 8 * t;
        const v4i x = *reinterpret_cast<const v4i *>(cstage + row * 128 + ((c16 ^ lrow) << 4));
        v4i o;  // undo the in-chunk rotation: (row >> 3) & 3 == t & 3
        o[0] = x[(0 + t) & 3];
        o[1] = x[(1 + t) & 3];
        o[2] = x[(2 + t) & 3];
        o[3] = x[(3 + t) & 3];
        const int m = m_w + row;
        if (FULL) {
          // (the staged form only runs on outputs of a dozen megabytes and more: streamed past the L2, they leave no
          //  dirty lines for the end-of-kernel write-back, which otherwise adds ~1.5 us before the next kernel starts)
          __builtin_nontemporal_store(o, reinterpret_cast<v4i_any *>(c + (int64_t)m * g.ldc + n));
        } else if (m < g.m && n < g.n) {
          store16(c + (int64_t)m * g.ldc + n, n, o);
        }
      };
      // the workgroup-shared form: wave w stores rows 32 w .. 32 w + 31 of the tile, 8 per instruction
      auto store_rows_wg = [&](int tt) {
        const int c16 = lane & 7, lrow = lane >> 3;
        const int n = n_tile + c16 * 16;
        const int row = lrow + 8 * (4 * (wm_id * 2 + wn_id) + tt);
        const v4i x = *reinterpret_cast<const v4i *>(cstage_wg + row * 128 + ((c16 ^ lrow) << 4));
        v4i o;  // undo the in-chunk rotation: (row >> 3) & 3 == tt
        o[0] = x[(0 + tt) & 3];
        o[1] = x[(1 + tt) & 3];
        o[2] = x[(2 + tt) & 3];
        o[3] = x[(3 + tt) & 3];
        const int m = m_tile + row;
        if (FULL) {
          *reinterpret_cast<v4i_any *>(c + (int64_t)m * g.ldc + n) = o;
        } else if (m < g.m && n < g.n) {
          store16(c + (int64_t)m * g.ldc + n, n, o);
        }
      };
      // any other workgroup-shared form: 16-byte chunks of the tile in row order, 256 at a time
      auto store_any = [&](int t) {
        constexpr int kChunks = 4 * TN;
        const int id = t * 256 + (wm_id * 2 + wn_id) * 64 + lane;
        const int row = id / kChunks, c16 = id - row * kChunks;
        const v4i o = *reinterpret_cast<const v4i *>(cstage_wg + row * epi_row_bytes<TN>() + c16 * 16);
        const int m = m_tile + row, n = n_tile + c16 * 16;
        if (FULL) {
          *reinterpret_cast<v4i_any *>(c + (int64_t)m * g.ldc + n) = o;
        } else if (m < g.m && n < g.n) {
          store16(c + (int64_t)m * g.ldc + n, n, o);
        }
      };
      constexpr int kPhases = kStageC ? 2 : 1, kJ = TM / kPhases;  // row blocks per pass over the channels
      // where this lane's dword of piece (i, q) goes in its staging row (see the layout above)
      int stage_off[(kStageC || kStageWG) ? TN * 4 : 1];
      if (kStageWG) {
  #pragma unroll
        for (int i = 0; i < TN; ++i)
  #pragma unroll
          for (int q = 0; q < 4; ++q)
            stage_off[i * 4 + q] = (wm_id * 32 * TM + r) * 128 + (((wn_id * 4 + 2 * i + (q >> 1)) ^ (r & 7)) << 4) +
                                   (((2 * q + h + (r >> 3)) & 3) << 2);
      }
      if (kStageC) {
  #pragma unroll
        for (int i = 0; i < TN; ++i)
  #pragma unroll
          for (int q = 0; q < 4; ++q)
            stage_off[i * 4 + q] = r * 128 + (((2 * i + (q >> 1)) ^ (r & 7)) << 4) + (((2 * q + h + (r >> 3)) & 3) << 2);
      }
      // per-channel constants of one piece (4 channels); the next piece's are requested before this piece's
      // arithmetic starts, so that the LDS latency is not paid once per piece
      struct Piece {
        v4i mult4, bias4, e4, zw4, ls4, pre4, c01, c23;
      };
      auto load_piece = [&](int blk) {
        Piece pc;
        const int i = (blk >> 2) % TN, q = blk & 3;
        int nb = n_w + i * 32 + q * 8 + h * 4;
        const int *pl = p + (nb - n_tile);
        pc.mult4 = *reinterpret_cast<const v4i *>(pl);
        pc.bias4 = pc.zw4 = pc.ls4 = pc.pre4 = pc.c01 = pc.c23 = v4i{0, 0, 0, 0};
        if (FAST) {
          pc.c01 = *reinterpret_cast<const v4i *>(p + TILE_N + 2 * (nb - n_tile));  // {lo, hi} x 2
          pc.c23 = *reinterpret_cast<const v4i *>(p + TILE_N + 2 * (nb - n_tile) + 4);
          pc.pre4 = *reinterpret_cast<const v4i *>(pl + 3 * TILE_N);
          pc.e4 = *reinterpret_cast<const v4i *>(pl + 4 * TILE_N);
          if (HAS_ZW) pc.zw4 = *reinterpret_cast<const v4i *>(pl + 5 * TILE_N);
        } else {
          pc.bias4 = *reinterpret_cast<const v4i *>(pl + TILE_N);
          pc.e4 = *reinterpret_cast<const v4i *>(pl + 2 * TILE_N);
          if (HAS_ZW) pc.zw4 = *reinterpret_cast<const v4i *>(pl + 3 * TILE_N);
          pc.ls4 = *reinterpret_cast<const v4i *>(pl + 4 * TILE_N);
  #pragma unroll
          for (int e = 0; e < 4; ++e) pc.bias4[e] = (int32_t)((uint32_t)pc.bias4[e] - ACC0);
        }
        return pc;
      };
      Piece next = load_piece(0);
  #pragma unroll
      for (int ph = 0; ph < kPhases; ++ph) {
  #pragma unroll
        for (int i = 0; i < TN; ++i) {
  #pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int nb = n_w + i * 32 + q * 8 + h * 4;
            const Piece pc = next;
            next = load_piece(i * 4 + q + 1);  // (wraps to piece 0 for the next pass; the arrays are padded)
            // (the staged form computes every channel of the padded tile and lets the stores check the bounds)
            if (!kStageC && !kStageWG && !kStageAny && nb >= g.n) continue;
            const v4i c2lo4 = v4i{pc.c01[0], pc.c01[2], pc.c23[0], pc.c23[2]};
            const v4i c2hi4 = v4i{pc.c01[1], pc.c01[3], pc.c23[1], pc.c23[3]};
  #pragma unroll
            for (int jj = 0; jj < kJ; ++jj) {
              const int j = ph * kJ + jj;
              int y[4];
              const int32_t a4[4] = {acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]};
              requant4(a4, rowsum[j], pc.mult4, c2lo4, c2hi4, pc.pre4, pc.bias4, pc.e4, pc.ls4, pc.zw4, y);
              const uint32_t packed = pack4(y[0], y[1], y[2], y[3]);
              if (kStageC) {
                *reinterpret_cast<uint32_t *>(cstage + j * 32 * 128 + stage_off[i * 4 + q]) = packed;
              } else if (kStageWG) {
                *reinterpret_cast<uint32_t *>(cstage_wg + j * 32 * 128 + stage_off[i * 4 + q]) = packed;
              } else if (kStageAny) {
                *reinterpret_cast<uint32_t *>(cstage_wg + (m_w - m_tile + j * 32 + r) * epi_row_bytes<TN>() + nb - n_tile) = packed;
              } else {
                const int m = m_w + j * 32 + r;
                if (m < g.m) store4(c + (int64_t)m * g.ldc + nb, nb, packed);
              }
            }
            if (kStageC && ph == 1 && (q & 1)) {  // the first half's eight store instructions, one per two pieces
              __builtin_amdgcn_sched_barrier(0);
              store_rows(i * 2 + (q >> 1));
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
      }
      if (kStageC) {
  #pragma unroll
        for (int t = 8; t < 16; ++t) store_rows(t);
      }
      if (kStageWG) {
        __syncthreads();
  #pragma unroll
        for (int tt = 0; tt < 4; ++tt) store_rows_wg(tt);
      }
      if (kStageAny) {
        __syncthreads();
  #pragma unroll
        for (int t = 0; t < TN * TM; ++t) store_any(t);
      }
    };
    if (full_tile) {
      body(std::true_type());
    } else {
      body(std::false_type());
    }
  } else {
    float *c = static_cast<float *>(g.c);
    const int32_t zx = din.zx;
    const uint32_t kzz = (uint32_t)dq.deep * (uint32_t)zx * (uint32_t)dq.zw0;
    // As for the int8 output, the accumulator layout (a lane holds 4 consecutive columns of 32 different rows) is
    // turned into whole 128-byte row segments before it meets global memory: per 32-column block the wave's
    // TM x 32 rows go through a wave-private LDS tile (row stride 144 bytes: the 16-byte writes of 8 consecutive
    // rows and the 16-byte reads along a row are both bank-conflict free) and leave as 8 rows x 128 B per store.
    constexpr int kRowB = kDeqStageRowBytes;
    const int lane = h * 32 + r;
    const int lr = lane >> 3, lc = lane & 7;
    const bool has_bias = dq.has_bias != 0;
    // The body exists three times, chosen once per tile instead of with branches around every output: full tile
    // without activation and with one input scale (no bounds compares, no clamps, the scale product hoisted), full
    // tile in general, ragged tile in general.
    // The general bodies clamp between bounds that are infinite where the reference makes no comparison: (-inf > d)
    // and (inf < d) are false for every d, NaN included, so no activation, ReLU and ReLU6 share one form.
    const bool with_act = dq.act == MI_ACT_RELU || dq.act == MI_ACT_RELU6;
    const float act_lo = with_act ? 0.0f : -__builtin_inff();
    const float act_hi = dq.act == MI_ACT_RELU6 ? 6.0f : __builtin_inff();
    auto body = [&](auto full_c, auto act_c, auto rows_c) {
      constexpr bool FULL = decltype(full_c)::value, ACT = decltype(act_c)::value, PER_ROW = decltype(rows_c)::value;
#pragma unroll
      for (int i = 0; i < TN; ++i) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int nb = n_w + i * 32 + q * 8 + h * 4;
          const int *pl = p + (nb - n_tile);
          const v4f ws4 = *reinterpret_cast<const v4f *>(pl);
          const v4i wsum4 = *reinterpret_cast<const v4i *>(pl + TILE_N);
          const v4f b4 = *reinterpret_cast<const v4f *>(pl + 2 * TILE_N);
          uint32_t corr[4];
          float s4[4];  // one input scale for the whole tensor: the scale product is the same for every row
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            corr[e] = kzz - (uint32_t)zx * (uint32_t)wsum4[e] - ACC0;
            s4[e] = __fmul_rn(din.sx, ws4[e]);
          }
#pragma unroll
          for (int j = 0; j < TM; ++j) {
            v4f o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              uint32_t v = (uint32_t)acc[i][j][q * 4 + e] + corr[e];
              if (HAS_ZW) v -= (uint32_t)dq.zw0 * (uint32_t)rowsum[j];
              float d = __fmul_rn(PER_ROW ? __fmul_rn(din.sxr[j], ws4[e]) : s4[e], (float)(int32_t)v);
              if (has_bias) d = __fadd_rn(d, b4[e]);
              if (ACT) {
                d = (act_lo > d) ? act_lo : d;
                d = (act_hi < d) ? act_hi : d;
              }
              o[e] = d;
            }
            *reinterpret_cast<v4f *>(cstage + (j * 32 + r) * kRowB + (q * 8 + h * 4) * 4) = o;
          }
        }
        const int n = n_w + i * 32 + lc * 4;
#pragma unroll
        for (int t = 0; t < TM * 4; ++t) {
          const int row = t * 8 + lr;
          const v4f v = *reinterpret_cast<const v4f *>(cstage + row * kRowB + lc * 16);
          const int m = m_w + row;
          if (!FULL && m < g.m && n < g.n && n + 4 > g.n) {
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (n + e < g.n) c[(int64_t)m * g.ldc + n + e] = v[e];
          } else if (FULL || (m < g.m && n < g.n)) {
            v4f_any *dst = reinterpret_cast<v4f_any *>(c + (int64_t)m * g.ldc + n);
            if (FAST) {  // in this epilogue the parameter selects non-temporal stores (see stream_out_hint)
              __builtin_nontemporal_store(v, dst);
            } else {
              *dst = v;
            }
          }
        }
      }
    };
    const bool full_tile = m_w + 32 * TM <= g.m && n_w + 32 * TN <= g.n;
    // (the common case, a full tile of a MatMul without activation and with one input scale, has a body of its own;
    //  per-row scales and activations share the general one)
    if (full_tile && !with_act && !dq.per_row) {
      body(std::true_type(), std::false_type(), std::false_type());
    } else if (full_tile) {
      body(std::true_type(), std::true_type(), std::true_type());
    } else {
      body(std::false_type(), std::true_type(), std::true_type());
    }
  }
}

template <int TN, int TM>
struct Frag {
  v4i w[TN], a[TM];
};

// Sums of the activation rows, which weights with zero points need: one v_mfma_i32_16x16x64_i8 for 32 bytes of K of 32 rows.
// In the fragment of a 32x32x32 product lane 32 h + r holds 16 bytes of row r; the 16x16x64 product takes lane 16 c + i as 16
// bytes of its column i.  Rows 16 .. 31 are then chunks c = 1 and 3 of columns 0 .. 15: four rows of its other operand with
// ones at chunks 0 and 2 add up rows 0 .. 15, four with ones at 1 and 3 the rest, and the sum of row r arrives in lane r.
// For gemm_ring.h: v_dot4, four for as many bytes, take 15 cycles each there and keep the wave from issuing anything else,
// while the matrix cores are idle for most of a small tile.  us with v_dot4 -> this (without zero points): 128 x 2048 x 1024
// 7.25 -> 6.05 (5.6), 400 x 2048 x 1024 7.45 -> 6.25 (5.7), 333 x 1024 x 1024 5.25 -> 4.9 (4.35), 128 x 4096 x 4096 in parts 11.0 ->
// 10.4 (9.4).  The loops that hide the v_dot4 behind their own products gain nothing and keep them: 128 x 128 tiles 24.0 -> 24.0,
// gemm_anyrow.hip 5.45 -> 5.5.
template <int TM>
struct RowSums {
  v4i sum[TM];
  int ones;
  __device__ __forceinline__ void clear(int lane) {
    const int i = lane & 15, c = lane >> 4;
    ones = (i >> 2) < 2 && (c & 1) == (i >> 2) ? 0x01010101 : 0;
#pragma unroll
    for (int j = 0; j < TM; ++j) sum[j] = v4i{0, 0, 0, 0};
  }
  // live: this lane's 16 bytes lie inside K
  __device__ __forceinline__ void add(const v4i (&a)[TM], bool live) {
    const int o = live ? ones : 0;
#pragma unroll
    for (int j = 0; j < TM; ++j) sum[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{o, o, o, o}, a[j], sum[j], 0, 0, 0);
  }
  __device__ __forceinline__ void get(int (&rowsum)[TM]) const {
#pragma unroll
    for (int j = 0; j < TM; ++j) rowsum[j] = sum[j][0];
  }
};

// The ring's loops (gemm_ring.h): up to two row tiles the weights stream past the L2s, which then keep the activations that every
// channel tile re-reads.  With more row tiles too many workgroups rely on finding them there.  us per launch, weights from HBM,
// plain -> streamed: one row tile, 128 x 12288 x 4096 18.4 -> 16.3, 128 x 11008 x 4096 17.6 -> 16.0; two, 256 x 12288 x 4096 26.3 -> 23.4,
// 128 x 4096 x 4096 11.8 -> 11.0; three, 300 x 5504 x 2048 (fp32) 13.9 -> 14.8; four, 197 x 768 x 3072 (fp32) 8.2 -> 9.4;
// thirty-two, 4096 x 768 x 3072 (fp32) 16.3 -> 22.0.
constexpr int kStreamRowTiles = 2;

// Launches of the K-block loops (gemm_kblock.hip, gemm_ring.hip), one per tile shape: T = 10 x TN + TM, the workgroup's
// tile being 64 TN channels x 64 TM rows.  requant: int8 output, fast2 form or not; otherwise fp32, `fast` = non-temporal
// stores.
int launch_gemm_kblock(int tile, bool requant, bool has_zw, bool fast, GemmArgs g, const RequantParams &rq,
                       const DequantParams &dq, hipStream_t stream);
int launch_gemm_ring(int tile, bool requant, bool has_zw, bool fast, GemmArgs g, const RequantParams &rq,
                     const DequantParams &dq, hipStream_t stream);
// The ring's loop with K split over `parts` workgroups a tile (gemm_split.hip): tiles 11, 12 and 22, int8 output only in the fast2
// form, fp32 only without weight zero points; space: what split_space gave.
int launch_gemm_split(int tile, int parts, bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq,
                      const DequantParams &dq, void *space, hipStream_t stream);
// 64 x 64 tiles over activation rows of any length, stride and address (gemm_anyrow.hip); g.k: bytes of K.
int launch_gemm_anyrow(bool requant, bool has_zw, bool fast, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                       hipStream_t stream);
// 32 x 32 tiles, or 64 channels x 32 rows, the K blocks dealt to the waves of a workgroup (gemm_short.hip).  tile: 10 x waves + blocks of 32
// channels, 41, 81 or 82; any: rows of any length at any address, end to end (lda == k), g.k: bytes of K.  int8 output only in the fast2
// form, fp32 never with non-temporal stores.
int launch_gemm_short(int tile, bool any, bool requant, bool has_zw, const GemmArgs &g, const RequantParams &rq, const DequantParams &dq,
                      hipStream_t stream);
// The same for a group whose members have blocked weights without zero points (and, for int8 output, the fast2 form).
int launch_gemm_kblock_group(int tile, GemmGroup<RequantParams> grp, hipStream_t stream);
int launch_gemm_kblock_group(int tile, bool fast, GemmGroup<DequantParams> grp, hipStream_t stream);
int launch_gemm_ring_group(int tile, GemmGroup<RequantParams> grp, hipStream_t stream);
int launch_gemm_ring_group(int tile, bool fast, GemmGroup<DequantParams> grp, hipStream_t stream);

}  // namespace mi
