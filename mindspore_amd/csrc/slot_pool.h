// Which calls on host tensors get page-locked slots (host_copy.hip), and when the memory comes and goes.  Host code only.
#pragma once

#include <stddef.h>

#include <mutex>

namespace mi {

// Slots is a set of slots with a member `next`, made by Slots::make(size) (null: no memory) and given back by Slots::free.  A set
// serves one call at a time; idle ones wait for the next call while a handle that makes such calls lives (add_user / drop_user).
//
// A set costs page-locked memory, about 200 us to allocate, touch and give back (where a process has the pages for the first time
// 256 KiB take 240, 2 MiB 1000).  It saves a tensor about 5 us and 15 per MiB.  So tensors go without until what they would have
// saved comes to the price of a set: a program of a few small calls, or one that makes a handle for each, pays nothing.
// us, a set in the first call -> this: first call of a process on 64 rows of 64 490 -> 65 (hipMemcpy 65); a call of a new handle and its
// destruction on 256 x 1024 x 1024 270 -> 110 (102), on 64 x 64 x 64 220 -> 75 (75).
// As many sets as callers have met at once, up to kMostSets; callers beyond go without.
template <typename Slots>
class SlotPool {
 public:
  static constexpr int kSizes = 2, kMostSets = 8;
  static constexpr float kPrice = 200.0f;  // us

  void add_user() {
    std::lock_guard<std::mutex> lock(mutex_);
    ++users_;
  }
  void drop_user() {  // the last one takes the idle sets with it, which are all there are
    Slots *idle = nullptr;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (--users_ > 0) return;
      for (Size &s : sizes_) {
        while (Slots *x = s.idle) {
          s.idle = x->next;
          x->next = idle;
          idle = x;
        }
        s = Size{};
      }
    }
    while (idle != nullptr) {
      Slots *next = idle->next;
      Slots::free(idle);
      idle = next;
    }
  }

  // For a tensor of a user's call; null: it goes without.  pageable() is asked only where there is a set to be had: a tensor that is
  // not needs none.
  template <typename F>
  Slots *take(int size, size_t bytes, F pageable) {
    Size &s = sizes_[size];
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (s.idle == nullptr) {
        if (s.made == kMostSets) return nullptr;
        s.forgone += 5.0f + 15.0f / (1 << 20) * (float)bytes;
        if (s.forgone < kPrice) return nullptr;
      }
    }
    const bool wanted = pageable();
    {
      std::lock_guard<std::mutex> lock(mutex_);
      if (wanted && s.idle != nullptr) {
        Slots *x = s.idle;
        s.idle = x->next;
        return x;
      }
      s.forgone = 0.0f;
      if (!wanted || s.made == kMostSets) return nullptr;
      ++s.made;
    }
    Slots *x = Slots::make(size);
    if (x == nullptr) {
      std::lock_guard<std::mutex> lock(mutex_);
      --s.made;
    }
    return x;
  }
  void give(int size, Slots *x) {
    std::lock_guard<std::mutex> lock(mutex_);
    x->next = sizes_[size].idle;
    sizes_[size].idle = x;
  }

 private:
  struct Size {
    Slots *idle = nullptr;
    int made = 0;
    float forgone = 0.0f;  // us
  };
  std::mutex mutex_;
  Size sizes_[kSizes];
  int users_ = 0;
};

}  // namespace mi
