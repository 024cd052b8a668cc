// Host tensors of the *_run_host calls, in and out of device memory through page-locked slots.
//
// hipMemcpy of 4 MiB of pageable memory takes 132 us in and 252 out; the bus needs 82 either way, and the host copies 4 MiB
// between pageable and page-locked memory in 54.  So the host copies a chunk into a slot while the device still reads the one
// before it, and on the way back takes a chunk out of its slot while the device writes the next.  The device's side is a copy
// kernel (a copy engine costs an event and its interrupt per chunk, 20 us; a launch costs 4), and what the host waits for is a
// word per part in the page-locked memory, written behind the part's bytes.
// MatMuls on host tensors, rows x K x N int8, us per call, hipMemcpy -> slots: 1024 x 4096 x 4096 412 -> 262,
// 2048 x 4096 x 4096 770 -> 511 to 555, 1000 x 256 x 4096 258 -> 150, 256 x 4096 x 1024 97 -> 70, 16 x 4096 x 4096 43 -> 25,
// 1 x 1024 x 1024 28.5 -> 17.  What is left is the bus, in and out one after the other.  slot_pool.h says which calls have slots.
// A copy in need not wait for the copy before it, which is of other bytes into another place, and starts while that still runs: one behind
// the other they leave the bus idle for the way to the host and back and the end of a launch, 2.5 us a chunk.  1024 x 4096 x 4096 262 -> 249,
// 2048 x 4096 x 4096 511 -> 490, 1000 x 256 x 4096 147 -> 131.
#include <hip/hip_ext.h>
#include <string.h>

#include <new>

#include "common.h"
#include "flag_wait.h"
#include "slot_pool.h"

namespace mi {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kWgBytes = 16384;  // 256 threads, four times 16 bytes each
// Page-locked memory of a call, cut into slots of a chunk each.  New pages cost 0.4 us per KiB once, so calls on small tensors get
// little; 1 MiB instead of 2 makes 262 us 303, 4 MiB 265.
constexpr size_t kRingBytes[2] = {256 << 10, 2 << 20};
constexpr int kMostSlots = 8;
constexpr int kOutWgs = 16;  // us at 4 MiB out: 16 149, 32 154, 64 159, 256 230 (1000 x 256 x 4096)

// Copies `n16` 16-byte words in parts of kWgBytes and says so in a flag per part.  TO_HOST: a flag follows the arrival of its
// part in host memory, and the workgroups, few enough to leave the bus to the first of them, take the parts in order, so that
// the host can empty the first slots while the last are being filled (with a workgroup per part all parts arrived at the end).
// Otherwise a flag says that its part has been read.
template <bool TO_HOST>
__global__ __launch_bounds__(256) void host_copy_kernel(const v4i *__restrict__ from, v4i *__restrict__ to, int n16, int wgs, uint32_t *flags,
                                                        uint32_t ticket) {
  constexpr int kPart = kWgBytes / 16;
  for (int part = blockIdx.x; part * kPart < n16; part += wgs) {
    const int first = part * kPart + threadIdx.x;
    v4i v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (first + 256 * j < n16) v[j] = __builtin_nontemporal_load(from + first + 256 * j);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (first + 256 * j < n16) to[first + 256 * j] = v[j];
    if (TO_HOST) __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flags + part, ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

struct HostSlots {
  int size = 0;               // kRingBytes[size] of
  char *data = nullptr;
  uint32_t *flags = nullptr;  // one word per kWgBytes of them
  uint32_t ticket = 0;        // of the last launch
  uint32_t pending[kMostSlots] = {};  // of the launch that uses the slot, 0: none
  HostSlots *next = nullptr;

  static HostSlots *make(int size) {
    HostSlots *s = new (std::nothrow) HostSlots();
    if (s == nullptr) return nullptr;
    const size_t flag_bytes = sizeof(uint32_t) * (kRingBytes[size] / kWgBytes);
    void *p = nullptr;
    if (hipHostMalloc(&p, kRingBytes[size] + flag_bytes, hipHostMallocCoherent | hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      delete s;
      return nullptr;
    }
    s->size = size;
    s->data = static_cast<char *>(p);
    s->flags = reinterpret_cast<uint32_t *>(s->data + kRingBytes[size]);
    memset(s->flags, 0, flag_bytes);
    return s;
  }
  static void free(HostSlots *s) {
    (void)hipHostFree(s->data);
    delete s;
  }
};

namespace {
SlotPool<HostSlots> g_pool;

// A transfer cut into chunks, of which chunk i goes through slot i % slots.
struct Chunks {
  size_t bytes, chunk;
  int64_t count;
  int slots;
  Chunks(size_t bytes_, size_t ring, size_t parts) : bytes(bytes_) {
    const size_t most = ring / parts;
    chunk = (bytes / parts + kWgBytes - 1) / kWgBytes * kWgBytes;
    chunk = chunk < 4 * kWgBytes ? 4 * kWgBytes : (chunk < most ? chunk : most);
    count = (int64_t)((bytes + chunk - 1) / chunk);
    slots = ring / chunk < kMostSlots ? (int)(ring / chunk) : kMostSlots;
  }
  int slot(int64_t i) const { return (int)(i % slots); }
  size_t at(int64_t i) const { return (size_t)i * chunk; }
  size_t size(int64_t i) const { return bytes - at(i) < chunk ? bytes - at(i) : chunk; }
  int wgs(size_t n) const { return (int)((n + kWgBytes - 1) / kWgBytes); }
  int first_flag(int slot) const { return slot * wgs(chunk); }
};

// A copy that may start before the launches in front of it are over.  hip_ext.h says of hipExtModuleLaunchKernel that GFX9 boards do not
// support the flag, and nothing of it for this call; here it is a hint.  With it as without, results hang on this alone: what is launched
// the ordinary way waits for everything launched before it on its stream, so a run, and through it the copies out, come behind all copies
// in; nobody else uses a copy's bytes at either end meanwhile (the slot is filled before the launch and again after its flags, the device's
// buffer is read by the run behind it, and the call before ended with its own run over).  No copy waits for another, and a later one
// may be over first: await_flags and drain() know that.
void launch_beside(const v4i *from, v4i *to, int n16, int parts, uint32_t *flags, uint32_t ticket) {
  void *list[] = {&from, &to, &n16, &parts, &flags, &ticket};
  (void)hipExtLaunchKernel(reinterpret_cast<const void *>(&host_copy_kernel<false>), dim3(parts), dim3(256), list, 0, nullptr, nullptr,
                           nullptr, hipExtAnyOrderLaunch);
}

// Launches the copies of chunks [i, i + n), whose slots lie side by side, on the null stream, where the run between the copies
// is.  dev: the chunk's first byte.  (The last up to 15 bytes past the end are inside the slot and inside the handle's buffer.)
int launch_chunks(HostSlots *s, const Chunks &c, int64_t i, int n, char *dev, bool in) {
  const size_t bytes = c.at(i + n - 1) + c.size(i + n - 1) - c.at(i);
  char *staged = s->data + c.at(c.slot(i));
  if (++s->ticket == 0) s->ticket = 1;
  const int n16 = (int)((bytes + 15) / 16), parts = c.wgs(bytes);
  uint32_t *flags = s->flags + c.first_flag(c.slot(i));
  v4i *there = reinterpret_cast<v4i *>(dev), *here = reinterpret_cast<v4i *>(staged);
  if (in && i > 0) {
    launch_beside(here, there, n16, parts, flags, s->ticket);
  } else if (in) {
    launch_kernel((host_copy_kernel<false>), dim3(parts), dim3(256), 0, nullptr, here, there, n16, parts, flags, s->ticket);
  } else {
    const int wgs = parts < kOutWgs ? parts : kOutWgs;
    launch_kernel((host_copy_kernel<true>), dim3(wgs), dim3(256), 0, nullptr, there, here, n16, wgs, flags, s->ticket);
  }
  MI_HIP_CHECK(hipGetLastError());
  for (int k = 0; k < n; ++k) s->pending[c.slot(i) + k] = s->ticket;
  return MI_OK;
}

// Until nothing that the null stream was given is under way: behind a launch of nothing the ordinary way, which waits for all copies.
hipError_t drain() {
  launch_kernel((host_copy_kernel<false>), dim3(1), dim3(256), 0, nullptr, nullptr, nullptr, 0, 1, nullptr, 0u);
  const hipError_t launched = hipGetLastError(), over = hipStreamSynchronize(nullptr);
  return launched != hipSuccess ? launched : over;
}

struct NullStream {  // as await_flags takes it
  int idle(bool *idle) {
    const hipError_t e = hipStreamQuery(nullptr);
    *idle = e == hipSuccess;
    if (e != hipErrorNotReady) MI_HIP_CHECK(e);
    return MI_OK;
  }
  int drain() {
    MI_HIP_CHECK(mi::drain());
    return MI_OK;
  }
};

// Until every workgroup that copies chunk i has said that it is done.
int await_chunk(HostSlots *s, const Chunks &c, int64_t i) {
  const int slot = c.slot(i);
  if (s->pending[slot] == 0) return MI_OK;
  const int rc = await_flags(s->flags + c.first_flag(slot), c.wgs(c.size(i)), s->pending[slot], NullStream());
  if (rc == kFlagMissing) {
    set_error("a copy between host and device ended without its result");
    return MI_ERROR;
  }
  if (rc == MI_OK) s->pending[slot] = 0;
  return rc;
}

// Page-locked memory, and anything else that the runtime knows, is hipMemcpy's: it needs no slots.
bool is_pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}
}  // namespace

HostCopyUser::~HostCopyUser() {
  if (used_) g_pool.drop_user();
}

HostCopies::HostCopies(HostCopyUser *user, size_t most_bytes) : user_(user), size_(most_bytes > kRingBytes[0] ? 1 : 0) {}

HostCopies::~HostCopies() {
  if (slots_ == nullptr) return;
  bool busy = false;  // (after an error: whoever has the slots next must not meet this call's copies)
  for (int i = 0; i < kMostSlots; ++i) busy = busy || slots_->pending[i] != 0;
  if (busy) (void)drain();
  for (int i = 0; i < kMostSlots; ++i) slots_->pending[i] = 0;
  g_pool.give(size_, slots_);
}

bool HostCopies::through_slots(const void *host, size_t bytes) {
  if (bytes == 0) return false;
  if (slots_ != nullptr) return is_pageable(host);
  if (!user_->used_) {
    user_->used_ = true;
    g_pool.add_user();
  }
  slots_ = g_pool.take(size_, bytes, [host] { return is_pageable(host); });
  return slots_ != nullptr;
}

int HostCopies::in(void *dev, const void *host, size_t bytes) {
  if (!through_slots(host, bytes)) {
    MI_HIP_CHECK(hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice));
    return MI_OK;
  }
  const Chunks c(bytes, kRingBytes[slots_->size], 4);  // a launch each: few and large
  int rc;
  for (int64_t i = 0; i < c.count; ++i) {
    if (i >= c.slots && (rc = await_chunk(slots_, c, i - c.slots)) != MI_OK) return rc;
    memcpy(slots_->data + c.at(c.slot(i)), static_cast<const char *>(host) + c.at(i), c.size(i));
    if ((rc = launch_chunks(slots_, c, i, 1, static_cast<char *>(dev) + c.at(i), true)) != MI_OK) return rc;
  }
  return MI_OK;
}

int HostCopies::out(void *host, const void *dev, size_t bytes) {
  if (!through_slots(host, bytes)) {
    MI_HIP_CHECK(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost));
    return MI_OK;
  }
  // Small chunks, and one launch for as many as there are slots at first, then for half of them whenever so many are empty.  (The
  // copies that came in through the same slots are over when these start: one stream.)
  const Chunks c(bytes, kRingBytes[slots_->size], 8);
  char *from = static_cast<char *>(const_cast<void *>(dev));
  const int half = c.slots / 2;
  for (uint32_t &p : slots_->pending) p = 0;
  int64_t asked = c.count < c.slots ? c.count : c.slots;
  int rc = launch_chunks(slots_, c, 0, (int)asked, from, false);
  for (int64_t i = 0; i < c.count && rc == MI_OK; ++i) {
    if ((rc = await_chunk(slots_, c, i)) != MI_OK) return rc;
    memcpy(static_cast<char *>(host) + c.at(i), slots_->data + c.at(c.slot(i)), c.size(i));
    if ((i + 1) % half == 0 && asked < c.count) {
      const int n = (int)(c.count - asked < half ? c.count - asked : half);
      rc = launch_chunks(slots_, c, asked, n, from + c.at(asked), false);
      asked += n;
    }
  }
  return rc;
}

}  // namespace mi
