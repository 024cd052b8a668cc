// The memory of split_space for the library's own streams: whose it is, and when it comes and goes.  Host code only.
#pragma once

#include <stddef.h>

#include <mutex>
#include <vector>

namespace mi {

// Memory has a type Stream; make(stream), device memory whose counters are zero before anything that the stream runs later (null:
// there is none); free(p), which may wait for all work on the device, and says whether it is gone.
//
// A stream gets its space when it is created, so that no run on it allocates: one of a few that are there for good (in a program of
// few sessions, streams then cost no memory and no time), otherwise one made for it.  Where there is none to be had it goes without.
// What was made stays for the next stream, since giving it back would make one session's end wait for the others' work; all of it is
// given back with the last stream.  So there are never more than there were streams at once.
template <typename Memory>
class SplitSpaces {
 public:
  typedef typename Memory::Stream Stream;

  void keep(int device, void *p) {  // a space that is there for good, its counters zero
    std::lock_guard<std::mutex> lock(mutex_);
    try {
      spaces_.push_back(Space{p, Stream(), device, kIdle, true});
    } catch (...) {  // (no host memory: one less)
    }
  }
  void enter(Stream stream, int device) {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (Space &s : spaces_) {
        if (s.state != kIdle || s.device != device) continue;
        s.stream = stream;
        s.state = kUsed;
        return;
      }
    }
    void *p = Memory::make(stream);
    if (p == nullptr) return;
    try {
      std::lock_guard<std::mutex> lock(mutex_);
      spaces_.push_back(Space{p, stream, device, kUsed, false});
    } catch (...) {
      (void)Memory::free(p);
    }
  }
  void *of(Stream stream) {
    std::lock_guard<std::mutex> lock(mutex_);
    Space *s = find(stream);
    return s != nullptr ? s->p : nullptr;
  }

  // The end of a stream: leave() before it is destroyed, with the space that it leaves (null: it has none) on to left() afterwards.
  // destroyed: it is gone, and not still there after an error; settled: nothing that ran on it still uses the space.
  void *leave(Stream stream) {
    std::lock_guard<std::mutex> lock(mutex_);
    Space *s = find(stream);
    if (s == nullptr) return nullptr;
    s->state = kLeaving;
    return s->p;
  }
  void left(void *p, bool destroyed, bool settled) {
    if (p == nullptr) return;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (Space &s : spaces_)
        if (s.p == p && s.state == kLeaving) s.state = !destroyed ? kUsed : settled ? kIdle : kNobodys;
    }
    while ((p = take_back()) != nullptr) {
      const bool gone = Memory::free(p);
      std::lock_guard<std::mutex> lock(mutex_);
      for (size_t i = 0; i < spaces_.size(); ++i) {
        if (spaces_[i].p != p || spaces_[i].state != kFreed) continue;
        if (gone) spaces_.erase(spaces_.begin() + (ptrdiff_t)i);
        else spaces_[i].state = kNobodys;
        break;
      }
      if (!gone) return;  // (the end of another stream tries again)
    }
  }

 private:
  enum State { kIdle, kUsed, kLeaving, kNobodys, kFreed };
  struct Space {
    void *p;
    Stream stream;
    int device;
    State state;
    bool for_good;
  };
  // One that was made and is to be given back, if no stream is left that has a space.
  void *take_back() {
    std::lock_guard<std::mutex> lock(mutex_);
    Space *made = nullptr;
    for (Space &s : spaces_) {
      if (s.state != kIdle && s.state != kNobodys) return nullptr;
      if (!s.for_good) made = &s;
    }
    if (made == nullptr) return nullptr;
    made->state = kFreed;
    return made->p;
  }
  Space *find(Stream stream) {
    for (Space &s : spaces_)
      if (s.state == kUsed && s.stream == stream) return &s;
    return nullptr;
  }
  std::mutex mutex_;
  std::vector<Space> spaces_;
};

}  // namespace mi
