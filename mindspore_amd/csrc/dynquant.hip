// DynamicQuant: fp32 -> int8 with scale / zero point taken from the min and max of the tensor, or of each of its rows.
// Bound by HBM for large tensors (5 bytes per value) and by the latency of one chain -- fetch, reduce, derive the
// parameters, quantise, store -- for small ones, so a thread requests all its values before it uses the first and
// keeps them in registers until the parameters are known:
//   dq_fused    : a tensor in one launch; the workgroups exchange their min and max through memory
//   dq_rows     : one scale per row, a wave or a workgroup per row (dq_long_rows: rows too long for registers)
//   dq_minmax + dq_quantize : tensors larger than the registers of the device, two launches and two reads
// Arithmetic: running min/max with the strict </> updates of CalculateMinMaxFp32 (reference mindspore/ccsrc/plugin/
// device/cpu/kernel/nnacl/int8/dynamic_quant_int8.c:19-27; a NaN is never selected); scale / zero point exactly as
// DynamicQuantCPUKernel::CalculatePerlayerScaleZp (mindspore/lite/src/litert/kernel/cpu/int8/dynamic_quant.cc:156-186:
// float range, float division, zero point in double); DoQuantizeFp32ToInt8 (.../nnacl/int8/
// quant_dtype_cast_int8.c:180-203: float reciprocal, float multiply, float add, round half away, clamp).
#include <float.h>

#include "common.h"

namespace mi {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kDqThreads = 256;
constexpr int kDqElemsPerThread = 16;

// NaN is no minimum or maximum: made quiet, since the hardware's minimum of a signalling NaN and a number is NaN.  (v_max, and half
// of a v_min3 and a v_max3: two instructions a value, where comparisons and selections take four and their wait states.)
__device__ __forceinline__ void upd(float v, float &lo, float &hi) {
  v = __builtin_canonicalizef(v);
  lo = __builtin_fminf(lo, v);
  hi = __builtin_fmaxf(hi, v);
}

// Minimum and maximum over the 64 lanes of a wave, in every lane: DPP steps inside each row of 16 lanes (quad_perm
// [1,0,3,2], quad_perm [2,3,0,1], row_ror:4, row_ror:8), then one lane per row is read back.
__device__ __forceinline__ void wave_minmax(float &lo, float &hi) {
#define MI_DPP_STEP(ctrl)                                                                                     \
  {                                                                                                           \
    const int l2 = __builtin_amdgcn_update_dpp(__float_as_int(lo), __float_as_int(lo), ctrl, 0xF, 0xF, false); \
    const int h2 = __builtin_amdgcn_update_dpp(__float_as_int(hi), __float_as_int(hi), ctrl, 0xF, 0xF, false); \
    lo = __int_as_float(l2) < lo ? __int_as_float(l2) : lo;                                                   \
    hi = __int_as_float(h2) > hi ? __int_as_float(h2) : hi;                                                   \
  }
  MI_DPP_STEP(0xB1)
  MI_DPP_STEP(0x4E)
  MI_DPP_STEP(0x124)
  MI_DPP_STEP(0x128)
#undef MI_DPP_STEP
  const float l = lo, h = hi;
#pragma unroll
  for (int row = 0; row < 4; ++row) {
    const float l2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l), row * 16));
    const float h2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(h), row * 16));
    lo = row == 0 || l2 < lo ? l2 : lo;
    hi = row == 0 || h2 > hi ? h2 : hi;
  }
}

template <int THREADS = 256>
__device__ __forceinline__ void block_minmax(float &lo, float &hi, float *slo, float *shi) {
  wave_minmax(lo, hi);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    slo[wave] = lo;
    shi[wave] = hi;
  }
  __syncthreads();
  lo = slo[0];
  hi = shi[0];
#pragma unroll
  for (int w = 1; w < THREADS / 64; ++w) {
    lo = slo[w] < lo ? slo[w] : lo;
    hi = shi[w] > hi ? shi[w] : hi;
  }
  __syncthreads();
}

__global__ __launch_bounds__(kDqThreads) void dq_minmax_kernel(const float *__restrict__ x, int64_t n,
                                                               float2 *__restrict__ partials) {
  __shared__ float slo[kDqThreads / 64], shi[kDqThreads / 64];
  float lo = FLT_MAX, hi = -FLT_MAX;
  const int64_t stride = (int64_t)gridDim.x * kDqThreads;
  const int64_t gtid = (int64_t)blockIdx.x * kDqThreads + threadIdx.x;
  if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
    const int64_t n4 = n >> 2;
    const v4f *x4 = reinterpret_cast<const v4f *>(x);
    int64_t i = gtid;
    for (; i + 3 * stride < n4; i += 4 * stride) {  // four independent 16-byte loads in flight per thread
      v4f v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = x4[i + j * stride];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        upd(v[j].x, lo, hi);
        upd(v[j].y, lo, hi);
        upd(v[j].z, lo, hi);
        upd(v[j].w, lo, hi);
      }
    }
    for (; i < n4; i += stride) {
      const v4f v = x4[i];
      upd(v.x, lo, hi);
      upd(v.y, lo, hi);
      upd(v.z, lo, hi);
      upd(v.w, lo, hi);
    }
    for (int64_t i = (n4 << 2) + gtid; i < n; i += stride) upd(x[i], lo, hi);
  } else {
    for (int64_t i = gtid; i < n; i += stride) upd(x[i], lo, hi);
  }
  block_minmax(lo, hi, slo, shi);
  if (threadIdx.x == 0) partials[blockIdx.x] = make_float2(lo, hi);
}

__device__ __forceinline__ int double_to_int_x86(double r) {
  // cvttsd2si semantics: NaN or out of range -> INT_MIN
  return (r >= -2147483648.0 && r <= 2147483647.0) ? (int)r : INT32_MIN;
}

__device__ __forceinline__ int8_t quant_one(float v, float inv, float zpf) {
  if (v == INFINITY) return 127;
  if (v == -INFINITY) return -128;
  const float t = __fadd_rn(__fmul_rn(v, inv), zpf);
  const float r = roundf(t);  // half away from zero, exact
  int q = (r >= -2147483648.0f && r < 2147483648.0f) ? (int)r : INT32_MIN;
  q = q < 127 ? q : 127;
  q = q > -128 ? q : -128;
  return (int8_t)q;
}

__device__ __forceinline__ int four_bytes(const int (&q)[4]) {
  const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)q[1], (uint32_t)q[0], 0x0c0c0400u);
  const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)q[3], (uint32_t)q[2], 0x0c0c0400u);
  return (int)__builtin_amdgcn_perm(p23, p01, 0x05040100u);
}

// Whether |t| < 2^20 for all values, given the least and the greatest of them: t does not fall as the value rises, and NaN is neither
// (infinities, and values that a broken scale throws out of range, are not).
__device__ __forceinline__ bool quantises_plainly(float lo, float hi, float inv, float zpf) {
  const float a = __fadd_rn(__fmul_rn(lo, inv), zpf), b = __fadd_rn(__fmul_rn(hi, inv), zpf);
  return __builtin_fabsf(a) < 1048576.0f && __builtin_fabsf(b) < 1048576.0f;
}

// Four such values -> four bytes, quant_one in a third of the instructions: adding the largest float below one half, with t's
// sign, and truncating rounds half away from zero exactly (a sum that should stay below the next integer stays there,
// t = k + 0.5 ties up to it).  The maximum of NaN and a number is the number, -128 as quant_one has it.
// Whether that may be is one question for the whole tensor (or run), and what it is otherwise one loop: asked for every four values,
// with the other answer beside each, a thread's values were 175 instructions a group to jump through, cold in the instruction
// cache at every launch, of which 42 are left.  us per launch from a graph, with that and comparisons for the minimum and maximum
// (see upd) / without the first / without both: 4096 x 768 6.75 / 6.6 / 6.35, 4096 x 3072 16.55 / 16.05 / 15.8, 600 x 4096 6.6 / 6.4 /
// 6.1, 2000 x 4096 11.3 / 10.85 / 10.7, 6000 x 5632 55.3 / 55.4 / 50.7; a scale per row, 2048 x 4096 8.37 / 8.28 / 8.24.
__device__ __forceinline__ int quant_four_plain(v4f v, float inv, float zpf) {
  int q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float t = __fadd_rn(__fmul_rn(v[e], inv), zpf);
    const float r = __fadd_rn(t, __builtin_copysignf(0x1.fffffep-2f, t));
    q[e] = (int)__builtin_fminf(__builtin_fmaxf(r, -128.0f), 127.0f);
  }
  return four_bytes(q);
}

__device__ __forceinline__ int quant_four(v4f v, float inv, float zpf) {
  int q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) q[e] = quant_one(v[e], inv, zpf);
  return four_bytes(q);
}

// scale and zero point from the tensor's min and max (CalculatePerlayerScaleZp, dynamic_quant.cc:156-186)
__device__ __forceinline__ void scale_and_zp(float lo, float hi, int symmetric, float *scale_f, int *zp) {
  *zp = 0;
  if (!symmetric) {
    float range = __fsub_rn(hi, lo);
    if (range <= 0) range = 0.01f;
    *scale_f = __fdiv_rn(range, 255.0f);
    *zp = double_to_int_x86(round(-128.0 - (double)lo / (double)*scale_f));
  } else {
    const float a = fabsf(hi), b = fabsf(lo);
    const float big = (a < b) ? b : a;
    *scale_f = __fdiv_rn(__fmul_rn(2.0f, big), 254.0f);
  }
}

// float4 at any float's address (the hardware loads 16 bytes from any 4-byte boundary in one instruction), and the
// four bytes it becomes, at any byte's address
typedef v4f v4f_any __attribute__((aligned(4)));
typedef int int_any __attribute__((aligned(1)));

__device__ __forceinline__ void upd4(v4f v, float &lo, float &hi) {
  upd(v.x, lo, hi);
  upd(v.y, lo, hi);
  upd(v.z, lo, hi);
  upd(v.w, lo, hi);
}

__device__ __forceinline__ void publish_params(mi_dq_params *p, float scale_f, int zp, float lo, float hi) {
  p->scale = (double)scale_f;
  p->scale_f = scale_f;
  p->zero_point = zp;
  p->real_min = lo;
  p->real_max = hi;
}

// The same to the host that is waiting for them, if one is: each word carries the run's ticket beside its value, so the
// stores need no order among themselves, and they leave before the quantising starts.
__device__ __forceinline__ void publish_to_host(const DqHostNote &note, float scale_f, int zp, float lo, float hi) {
  if (note.ticket == 0) return;
  const uint32_t v[kDqHostWords] = {__float_as_uint(scale_f), (uint32_t)zp, __float_as_uint(lo), __float_as_uint(hi)};
#pragma unroll
  for (int i = 0; i < kDqHostWords; ++i)
    __hip_atomic_store(note.words + i, (uint64_t)note.ticket << 32 | v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The whole of DynamicQuant in one launch: a workgroup keeps its share of the tensor (G float4 per thread, all of them
// requested before the first is used) in registers, publishes its min and max, waits for those of the other
// workgroups and quantises from the registers.  The tensor crosses HBM once, and a second launch and its re-read are
// saved for one exchange through memory.
//
// The exchange: workgroup s leaves its min and its max in slot s, each beside the launch's tag in one 64-bit word that either
// arrives whole or not at all, so no fence is needed and a word of an earlier launch is never taken for one of this.  Every
// launch fills all kDqSlots slots -- workgroup b takes b, b + W, .. for W workgroups, of which the first W are waited for --
// so a tag that comes round again after 2^31 launches finds none of its kind.  The host numbers the launches, except those
// that may be captured: a replay repeats its arguments, so there the number stands in memory (`replays`), and workgroup 0
// raises it when it has found the tag in every slot in use, hence after the last workgroup has read it.
//
// Launches on one handle are ordered by their stream.  Should two overlap, they disturb each other and no later one.  For
// numbers from memory: a workgroup that has given up waiting raises the number past its own tag too, and one that has not has
// seen its tag in slot 0, whose writer raises it, so in the end it is past every tag that was left in a slot.
//
// (Slots without tags that were emptied in turn, whose turn it was in a word per slot, took 0.2 us more; two 8-byte loads per slot
// instead of one of 16 0.3 to 0.7.)
//
// A workgroup looks at the slots for the first time when the others' words can be there (400 to 700 ns after its own, more with more
// values a workgroup, whose arrival spreads further).  A look that comes too early costs its whole way to memory and back, and 256
// workgroups looking over and over get in the way of the words they look for.  us per launch from a graph, first look at once / after
// this pause / twice it: 8 x 4096 4.15 / 3.93 / 4.4, 8 x 11008 4.7 / 4.15 / 4.5, 197 x 768 4.33 / 3.95 / 4.4, 197 x 3072 6.5 / 5.5 / 5.8,
// 481 x 2304 6.6 / 5.7, 4096 x 768 8.0 / 6.85, 4096 x 3072 17.2 / 16.55; with pauses between looks too 1 to 3 % more, with two or three
// looks on their way at once 0.4 to 0.7 us more than without any.
//
// The wait is bounded: workgroups that are not resident together (the device is shared) are not waited for for ever; a
// workgroup that has waited `patience` ticks of the 100 MHz counter reads the whole tensor itself.
constexpr int kDqSlots = kDqFusedMost;
constexpr uint32_t kDqPatience = 20000;  // 200 us
constexpr int kAgentScope = 16;  // cache policy of a load from the device's coherence point (sc1)
struct DqSlots {
  unsigned long long replays;
  uint64_t pad;
  uint64_t range[kDqSlots][2];  // {min, max}, each below its tag
};
static_assert(sizeof(DqSlots) == kDqSlotBytes, "what the handle allocates and fills with zeros");

template <int T, int G>
__global__ __launch_bounds__(T) void dq_fused_kernel(const float *__restrict__ x, int64_t n, int symmetric,
                                                     DqSlots *slots, uint32_t launch, uint32_t patience, int wgs, DqHostNote note,
                                                     mi_dq_params *__restrict__ params, int8_t *__restrict__ q) {
  __shared__ float slo[T / 64], shi[T / 64], all[2];
  __shared__ int late_wg;
  const int tid = threadIdx.x, w = blockIdx.x;  // of wgs
  const int64_t n4 = n >> 2, first = (int64_t)w * (T * G) + tid;
  const v4f_any *x4 = reinterpret_cast<const v4f_any *>(x);
  const bool counted = launch == 0;  // the number of this launch stands in memory
  unsigned long long replay = 0;
  if (counted && wgs > 1 && tid < 64)
    replay = __hip_atomic_load(&slots->replays, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  v4f v[G];
  float lo = FLT_MAX, hi = -FLT_MAX;
  if (n4 > 0) {
#pragma unroll
    for (int j = 0; j < G; ++j) {  // past the end: the last group again, which changes neither minimum nor maximum
      const int64_t i = first + j * T;
      v[j] = __builtin_nontemporal_load(x4 + (i < n4 ? i : n4 - 1));
    }
#pragma unroll
    for (int j = 0; j < G; ++j) upd4(v[j], lo, hi);
  }
  float tail = 0.0f;  // the up to three values past the last whole group
  const int64_t ti = (n4 << 2) + tid;
  const bool has_tail = w == 0 && ti < n;
  if (has_tail) {
    tail = x[ti];
    upd(tail, lo, hi);
  }
  if (wgs == 1) {
    block_minmax<T>(lo, hi, slo, shi);
  } else {
    wave_minmax(lo, hi);
    if ((tid & 63) == 0) {
      slo[tid >> 6] = lo;
      shi[tid >> 6] = hi;
    }
    __syncthreads();
    if (tid < 64) {  // one wave speaks for the workgroup
#pragma unroll
      for (int i = 0; i < T / 64; ++i) {
        lo = slo[i] < lo ? slo[i] : lo;
        hi = shi[i] > hi ? shi[i] : hi;
      }
      const uint32_t tag = counted ? (uint32_t)replay | kDqReplayed : launch;
      const uint64_t my_lo = (uint64_t)tag << 32 | __float_as_uint(lo), my_hi = (uint64_t)tag << 32 | __float_as_uint(hi);
      for (int s = w + tid * wgs; s < kDqSlots; s += 64 * wgs) {
        __hip_atomic_store(&slots->range[s][0], my_lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&slots->range[s][1], my_hi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __builtin_amdgcn_s_sleep(T * G <= 512 ? 14 : T * G <= 2048 ? 20 : 24);  // (see above)
      const uint64_t began = __builtin_amdgcn_s_memrealtime();
      bool late = false;
      // (16 bytes a load, past the caches of this XCD: two words that need not belong together, hence a tag in each)
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(slots->range, (short)0, sizeof(slots->range), 0x00020000);
      typedef uint32_t v4u __attribute__((ext_vector_type(4)));
      v4u got[kDqSlots / 64];
      while (true) {
#pragma unroll
        for (int i = 0; i < kDqSlots / 64; ++i) {
          const int s = tid + i * 64;
          got[i] = v4u{(uint32_t)my_lo, tag, (uint32_t)my_hi, tag};
          if (i * 64 < wgs)
            got[i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * (s < wgs ? s : w), 0, kAgentScope));
        }
        asm volatile("" ::: "memory");  // (requested anew every time round)
        bool missing = false;
#pragma unroll
        for (int i = 0; i < kDqSlots / 64; ++i) missing |= got[i][1] != tag || got[i][3] != tag;
        if (!__any(missing)) break;
        if (__builtin_amdgcn_s_memrealtime() - began > patience) {
          late = true;
          break;
        }
      }
      if (counted && tid == 0 && (w == 0 || late)) atomicMax(&slots->replays, replay);
      if (!late) {
#pragma unroll
        for (int i = 0; i < kDqSlots / 64; ++i) {
          const float l2 = __uint_as_float(got[i][0]), h2 = __uint_as_float(got[i][2]);
          lo = l2 < lo ? l2 : lo;
          hi = h2 > hi ? h2 : hi;
        }
        wave_minmax(lo, hi);
      }
      if (tid == 0) {
        all[0] = lo;
        all[1] = hi;
        late_wg = late;
      }
    }
    __syncthreads();
    lo = all[0];
    hi = all[1];
    if (late_wg) {
      for (int64_t i = tid; i < n4; i += T) upd4(x4[i], lo, hi);
      if (ti < n) upd(x[ti], lo, hi);
      block_minmax<T>(lo, hi, slo, shi);
    }
  }
  float scale_f;
  int zp;
  scale_and_zp(lo, hi, symmetric, &scale_f, &zp);
  if (w == 0 && tid == 0) {
    publish_to_host(note, scale_f, zp, lo, hi);
    publish_params(params, scale_f, zp, lo, hi);
  }
  const float inv = __fdiv_rn(1.0f, scale_f);
  const float zpf = (float)zp;
  if (quantises_plainly(lo, hi, inv, zpf)) {
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int64_t i = first + j * T;
      if (i < n4) *reinterpret_cast<int_any *>(q + 4 * i) = quant_four_plain(v[j], inv, zpf);
    }
  } else {  // (from memory again: with the registers, whose numbers are constants, there would be G copies of it)
#pragma unroll 1
    for (int64_t i = first; i < n4 && i < first + (int64_t)G * T; i += T)
      *reinterpret_cast<int_any *>(q + 4 * i) = quant_four(x4[i], inv, zpf);
  }
  if (has_tail) q[ti] = quant_one(tail, inv, zpf);
}

__global__ __launch_bounds__(kDqThreads) void dq_quantize_kernel(const float *__restrict__ x, int64_t n,
                                                                 int symmetric,
                                                                 const float2 *__restrict__ partials, int nparts, DqHostNote note,
                                                                 mi_dq_params *__restrict__ params,
                                                                 int8_t *__restrict__ q) {
  __shared__ float slo[kDqThreads / 64], shi[kDqThreads / 64];
  // request this thread's 16 values first: they arrive while the partials are reduced and the scale is derived
  const int64_t base = ((int64_t)blockIdx.x * kDqThreads + threadIdx.x) * kDqElemsPerThread;
  const bool aligned = ((reinterpret_cast<uintptr_t>(x) & 15) == 0) && ((reinterpret_cast<uintptr_t>(q) & 15) == 0);
  const bool fast = aligned && base + kDqElemsPerThread <= n;
  v4f xv[4];
  {
    // never predicated: a thread without a full group of its own re-reads the first one (n >= 16 on this path)
    const int64_t safe = fast ? base : 0;
    const v4f *x4 = reinterpret_cast<const v4f *>(x + (aligned && n >= kDqElemsPerThread ? safe : 0));
    if (aligned && n >= kDqElemsPerThread) {
#pragma unroll
      for (int j = 0; j < 4; ++j) xv[j] = x4[j];
    }
  }

  float lo = FLT_MAX, hi = -FLT_MAX;
  for (int i = threadIdx.x; i < nparts; i += kDqThreads) {
    const float2 p = partials[i];
    lo = p.x < lo ? p.x : lo;
    hi = p.y > hi ? p.y : hi;
  }
  block_minmax(lo, hi, slo, shi);

  float scale_f;
  int zp;
  scale_and_zp(lo, hi, symmetric, &scale_f, &zp);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    publish_to_host(note, scale_f, zp, lo, hi);
    publish_params(params, scale_f, zp, lo, hi);
  }
  const float inv = __fdiv_rn(1.0f, scale_f);
  const float zpf = (float)zp;

  if (base >= n) return;
  if (fast && quantises_plainly(lo, hi, inv, zpf)) {
    typedef int v4i __attribute__((ext_vector_type(4)));
    v4i o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = quant_four_plain(xv[j], inv, zpf);
    *reinterpret_cast<v4i *>(q + base) = o;
  } else {
    const int64_t end = base + kDqElemsPerThread < n ? base + kDqElemsPerThread : n;
    for (int64_t i = base; i < end; ++i) q[i] = quant_one(x[i], inv, zpf);
  }
}

// DynamicQuant with preferred axes (one scale / zero point per segment): after the preferred axes lead, the tensor is
// `segments` contiguous runs of `unit` elements (DynamicQuantCPUKernel::ReSize / CalculateMinMax / QuantData,
// mindspore/lite/src/litert/kernel/cpu/int8/dynamic_quant.cc:59-94,118-143,236-246; scale and zero point per segment
// as CalculatePerChannelScaleZp :188-218, the same formulas as the per-tensor case).  T threads per run keep it in
// registers, G float4 each, all requested before the first is used: one read of the tensor, and enough of it in
// flight.  T = 64: a wave per run, four runs per workgroup, no barrier; otherwise a workgroup per run.
template <int T, int G>
__global__ __launch_bounds__(T == 64 ? 256 : T) void dq_rows_kernel(const float *__restrict__ x, int64_t segments,
                                                                    int unit, int symmetric,
                                                                    mi_dq_params *__restrict__ params,
                                                                    int8_t *__restrict__ q) {
  const int tid = T == 64 ? threadIdx.x & 63 : threadIdx.x;
  const int64_t seg = T == 64 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : (int64_t)blockIdx.x;
  if (seg >= segments) return;  // a whole wave, and a whole workgroup where T > 64
  const float *xs = x + seg * unit;
  int8_t *qs = q + seg * unit;
  const int n4 = unit >> 2;
  const v4f_any *x4 = reinterpret_cast<const v4f_any *>(xs);
  v4f v[G];
  float lo = FLT_MAX, hi = -FLT_MAX;
  if (n4 > 0) {
#pragma unroll
    for (int j = 0; j < G; ++j) {  // past the end: the last group again
      const int i = tid + j * T;
      v[j] = __builtin_nontemporal_load(x4 + (i < n4 ? i : n4 - 1));
    }
#pragma unroll
    for (int j = 0; j < G; ++j) upd4(v[j], lo, hi);
  }
  float tail = 0.0f;  // the up to three values past the last whole group
  const int ti = (n4 << 2) + tid;
  if (ti < unit) {
    tail = xs[ti];
    upd(tail, lo, hi);
  }
  if constexpr (T == 64) {
    wave_minmax(lo, hi);
  } else {
    __shared__ float slo[T / 64], shi[T / 64];
    block_minmax<T>(lo, hi, slo, shi);
  }
  float scale_f;
  int zp;
  scale_and_zp(lo, hi, symmetric, &scale_f, &zp);
  if (tid == 0) publish_params(params + seg, scale_f, zp, lo, hi);
  const float inv = __fdiv_rn(1.0f, scale_f);
  const float zpf = (float)zp;
  if (quantises_plainly(lo, hi, inv, zpf)) {
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int i = tid + j * T;
      if (i < n4) *reinterpret_cast<int_any *>(qs + 4 * i) = quant_four_plain(v[j], inv, zpf);
    }
  } else {
#pragma unroll 1
    for (int i = tid; i < n4; i += T) *reinterpret_cast<int_any *>(qs + 4 * i) = quant_four(x4[i], inv, zpf);
  }
  if (ti < unit) qs[ti] = quant_one(tail, inv, zpf);
}

// Runs too long for registers: a workgroup per run, two sweeps.
__global__ __launch_bounds__(1024) void dq_long_rows_kernel(const float *__restrict__ x, int64_t segments, int64_t unit,
                                                            int symmetric, mi_dq_params *__restrict__ params,
                                                            int8_t *__restrict__ q) {
  __shared__ float slo[16], shi[16];
  const int tid = threadIdx.x;
  const float *xs = x + (int64_t)blockIdx.x * unit;
  int8_t *qs = q + (int64_t)blockIdx.x * unit;
  const int64_t n4 = unit >> 2;
  const v4f_any *x4 = reinterpret_cast<const v4f_any *>(xs);
  float lo = FLT_MAX, hi = -FLT_MAX;
  int64_t i = tid;
  for (; i + 3 * 1024 < n4; i += 4 * 1024) {
    v4f v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = x4[i + j * 1024];
#pragma unroll
    for (int j = 0; j < 4; ++j) upd4(v[j], lo, hi);
  }
  for (; i < n4; i += 1024) upd4(x4[i], lo, hi);
  const int64_t ti = (n4 << 2) + tid;
  if (ti < unit) upd(xs[ti], lo, hi);
  block_minmax<1024>(lo, hi, slo, shi);
  float scale_f;
  int zp;
  scale_and_zp(lo, hi, symmetric, &scale_f, &zp);
  if (tid == 0) publish_params(params + blockIdx.x, scale_f, zp, lo, hi);
  const float inv = __fdiv_rn(1.0f, scale_f);
  const float zpf = (float)zp;
  const bool plain = quantises_plainly(lo, hi, inv, zpf);
  for (int64_t k = tid; k < n4; k += 1024)
    *reinterpret_cast<int_any *>(qs + 4 * k) = plain ? quant_four_plain(x4[k], inv, zpf) : quant_four(x4[k], inv, zpf);
  if (ti < unit) qs[ti] = quant_one(xs[ti], inv, zpf);
}

template <int T, int G>
static void launch_rows(const float *x, int64_t segments, int unit, int symmetric, mi_dq_params *params, int8_t *q,
                        hipStream_t stream) {
  const int64_t blocks = T == 64 ? (segments + 3) / 4 : segments;
  launch_kernel((dq_rows_kernel<T, G>), dim3((unsigned)blocks), dim3(T == 64 ? 256 : T), 0, stream, x, segments,
                unit, symmetric, params, q);
}

int launch_dynquant_segments(const float *x, int64_t segments, int64_t unit, int symmetric, mi_dq_params *params,
                             int8_t *q, hipStream_t stream) {
  if (segments > 0x7fffffff) {
    set_error("dynquant: too many segments");
    return MI_PARAM_INVALID;
  }
  // A wave per run where there are enough short runs to fill the device with waves; otherwise more threads per run, for
  // few runs to shorten each thread's chain and for long ones to have 2 to 6 loads of 16 bytes per thread.  us per
  // launch, before (one wave per run, two sweeps) -> now: 8 x 4096 11.6 -> 2.9, 8 x 11008 28.0 -> 3.6,
  // 512 x 4096 14.8 -> 4.7, 4096 x 768 6.7 -> 5.2, 2048 x 4096 21.8 -> 8.2 (5.1 TB/s), 2048 x 11008 60.4 -> 19.9
  // (5.7 TB/s; a copy reaches 4.9).  2048 x 4096 takes 10.8 with a wave and 10.1 with 512 threads per run, 197 x 768
  // 3.0 with a wave and 2.7 with 256 threads, 4096 x 768 6.6 with 256 threads.
  const int64_t n4 = unit >> 2;
#define MI_DQ_ROWS(T, G) launch_rows<T, G>(x, segments, (int)unit, symmetric, params, q, stream)
  if (n4 <= 64) MI_DQ_ROWS(64, 1);
  else if (n4 <= 256 && segments >= 512) {
    if (n4 <= 128) MI_DQ_ROWS(64, 2);
    else if (n4 <= 192) MI_DQ_ROWS(64, 3);
    else MI_DQ_ROWS(64, 4);
  }
  else if (n4 <= 256) MI_DQ_ROWS(256, 1);
  else if (n4 <= 1024 && segments >= 256) {
    if (n4 <= 512) MI_DQ_ROWS(256, 2);
    else if (n4 <= 768) MI_DQ_ROWS(256, 3);
    else MI_DQ_ROWS(256, 4);
  }
  else if (n4 <= 1024) MI_DQ_ROWS(512, 2);
  else if (n4 <= 2048) MI_DQ_ROWS(512, 4);
  else if (n4 <= 3072) MI_DQ_ROWS(512, 6);
  else if (n4 <= 4096) MI_DQ_ROWS(512, 8);
  else if (n4 <= 16384) MI_DQ_ROWS(1024, 16);
  else
    launch_kernel(dq_long_rows_kernel, dim3((unsigned)segments), dim3(1024), 0, stream, x, segments, unit, symmetric,
                  params, q);
#undef MI_DQ_ROWS
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

template <int T, int G>
static void launch_fused(const float *x, int64_t n, int symmetric, void *slots, uint32_t launch, const DqHostNote &note,
                         mi_dq_params *params, int8_t *q, hipStream_t stream) {
  const int64_t want = ((n >> 2) + T * G - 1) / (T * G);
  const int wgs = want < 1 ? 1 : (int)want;
  launch_kernel((dq_fused_kernel<T, G>), dim3(wgs), dim3(T), 0, stream, x, n, symmetric,
                static_cast<DqSlots *>(slots), launch, kDqPatience, wgs, note, params, q);
}

int launch_dynquant(const float *x, int64_t n, int symmetric, float2 *partials, void *slots, uint32_t launch,
                    const DqHostNote &note, mi_dq_params *params, int8_t *q, hipStream_t stream) {
  // One launch as long as the tensor fits the registers of one workgroup per CU.  Up to 8192 values one workgroup is
  // faster than any exchange (about 0.9 us); from there on as many workgroups as there are slots, with the fewest
  // values per thread that allows: what counts at these sizes is the latency of each thread's chain.  us per tensor,
  // before (up to 24576 values one workgroup, else two launches) -> now: 4096 3.9 -> 2.9, 16384 5.9 -> 3.7,
  // 32768 7.2 -> 4.2, 88064 7.4 -> 4.4, 300000 7.7 -> 5.0, 1 M 8.0 -> 5.6, 4096 x 768 11.3 -> 8.9,
  // 2048 x 4096 20.0 -> 13.5, 4096 x 3072 26.9 -> 17.5, 2048 x 11008 40.8 -> 26.7.  (Since then the exchange and the quantising have
  // become quicker, see above: 32768 3.9, 88064 4.0, 4096 x 768 6.35, 4096 x 3072 15.8.)
  const int64_t n4 = n >> 2;
#define MI_DQ_FUSED(T, G)                                                        \
  do {                                                                           \
    launch_fused<T, G>(x, n, symmetric, slots, launch, note, params, q, stream); \
    MI_HIP_CHECK(hipGetLastError());                                             \
    return MI_OK;                                                                \
  } while (0)
  constexpr int64_t kMost = kDqFusedMost;
  if (n4 <= 256) MI_DQ_FUSED(256, 1);
  if (n4 <= 512 * 2) MI_DQ_FUSED(512, 2);
  if (n4 <= 512 * 4) MI_DQ_FUSED(512, 4);
  if (n4 <= kMost * 256) MI_DQ_FUSED(256, 1);
  if (n4 <= kMost * 512) MI_DQ_FUSED(512, 1);
  if (n4 <= kMost * 256 * 4) MI_DQ_FUSED(256, 4);
  if (n4 <= kMost * 512 * 4) MI_DQ_FUSED(512, 4);
  if (n4 <= kMost * 1024 * 3) MI_DQ_FUSED(1024, 3);
  if (n4 <= kMost * 1024 * 6) MI_DQ_FUSED(1024, 6);
  if (n4 <= kMost * 1024 * 8) MI_DQ_FUSED(1024, 8);
  if (n4 <= kMost * 1024 * 12) MI_DQ_FUSED(1024, 12);
  if (n4 <= kMost * 1024 * 16) MI_DQ_FUSED(1024, 16);
  if (n4 <= kMost * 1024 * 24) MI_DQ_FUSED(1024, 24);
#undef MI_DQ_FUSED
  const int64_t per_block = (int64_t)kDqThreads * kDqElemsPerThread;
  int64_t want = (n + per_block - 1) / per_block;
  // pass 1: at most one workgroup per partial a thread of pass 2 reads in a single step
  const int64_t want1 = (want + 2) / 3;
  const int nparts = (int)(want1 < 1 ? 1 : (want1 > kDqThreads ? kDqThreads : want1));
  launch_kernel(dq_minmax_kernel, dim3(nparts), dim3(kDqThreads), 0, stream, x, n, partials);
  MI_HIP_CHECK(hipGetLastError());
  const int64_t qblocks = want < 1 ? 1 : want;
  if (qblocks > 0x7fffffff) {
    set_error("dynquant: tensor too large");
    return MI_PARAM_INVALID;
  }
  launch_kernel(dq_quantize_kernel, dim3((unsigned)qblocks), dim3(kDqThreads), 0, stream, x, n, symmetric,
                partials, nparts, note, params, q);
  MI_HIP_CHECK(hipGetLastError());
  return MI_OK;
}

}  // namespace mi
