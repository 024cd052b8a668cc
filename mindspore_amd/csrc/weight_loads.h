// Where the K-block GEMM loops (gemm_kblock.hip, gemm_ring.hip) read the packed weights.  Plain integer arithmetic, so that
// the byte ranges can be checked on the host for every tile shape (tests/test_weight_loads.py).
#pragma once

#if defined(__HIPCC__)
#define MI_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define MI_HOST_DEVICE inline
#endif

namespace mi {

// The groups of 16 channels that one wave of a tile loads: wave w of a tile of 64 TN channels starting at n0 takes TN of them.
// The packed weights end at n rounded up to `pad` channels.  Where `pad` is no multiple of the tile, a wave's groups can lie
// past that end, partly or wholly; it then loads the last group that exists in their place, whose products reach only
// channels that are never stored.  (The range check of a buffer load does not serve here: the group is in the load's scalar
// offset, which the check leaves out.)
template <int TN>
struct WaveWeightGroups {
  int first;   // the wave's first group (or the last one that exists)
  int inside;  // groups from there on that exist, 1 .. TN
  MI_HOST_DEVICE WaveWeightGroups(int n, int n0, int wave, int pad) {
    const int groups = (n + pad - 1) / pad * pad / 16;
    first = n0 / 16 + wave * TN;
    inside = TN;
    if (pad % (64 * TN) != 0) {
      first = first < groups ? first : groups - 1;
      inside = groups - first < TN ? groups - first : TN;
    }
  }
  MI_HOST_DEVICE int group(int i) const { return i < inside ? i : inside - 1; }  // of the wave's i-th, counted from `first`
};

// Byte offset, from the wave's first group, of the loader instruction that fetches half `half` of group `group` in K block kb.
// Blocked copy: 1 KiB of 16 channels x 64 bytes of K, front to back (16 bytes per lane); k64 = k_pad / 64.
MI_HOST_DEVICE int blocked_weight_offset(int group, int half, int k64, int kb) { return (group * k64 + 2 * kb + half) * 1024; }
// Row-major: 8 rows x 128 bytes of K (a lane adds (lane / 8) * ldw and a 16-byte chunk below 128).
MI_HOST_DEVICE int row_major_weight_offset(int group, int half, int ldw, int kb) { return (16 * group + 8 * half) * ldw + 128 * kb; }

}  // namespace mi
