// Which calls on host tensors get page-locked slots (host_copy.hip), and when the memory comes and goes.  Host code only.
#pragma once

#include <stddef.h>

#include <mutex>

namespace mi {

// Slots is a set of slots with a member `next`, made by Slots::make(size) (null: no memory) and given back by Slots::free.  A set
// serves one call at a time; idle ones wait for the next call while a handle that makes such calls lives (add_user / drop_user).
//
// A set costs page-locked memory: us to allocate, touch and free, 256 KiB 80 + 110 + 50, 2 MiB 60 + 880 + 50, and about 200 where the
// process has had and given back the pages before.  It saves a tensor about 5 us and 15 per MiB.  So tensors go without until
// what they would have saved comes to the price of a set: a program of a few calls, or one that makes a handle for each, pays
// nothing, and no program more than it would have saved by then.  (The first call of a process on 64 rows of 64 took 490 us
// where it made slots, 65 without; on 1024 x 1024 640 and 465; handles of a single call on 256 x 1024 x 1024 and their destruction
// 270 and 102.)
// As many sets as callers have met at once, up to kMostSets; callers beyond go without.
template <typename Slots>
class SlotPool {
 public:
  static constexpr int kSizes = 2, kMostSets = 8;
  static constexpr float kPrice[kSizes] = {250.0f, 1000.0f}, kPriceAgain = 200.0f;  // us

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
        s.made = 0;
        s.forgone = 0.0f;
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
        if (s.forgone < (s.made < s.most ? kPriceAgain : kPrice[size])) return nullptr;
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
      if (++s.made > s.most) s.most = s.made;
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
    int made = 0, most = 0;  // now, ever
    float forgone = 0.0f;  // us
  };
  std::mutex mutex_;
  Size sizes_[kSizes];
  int users_ = 0;
};

}  // namespace mi
