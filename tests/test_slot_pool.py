"""Which calls on host tensors get page-locked slots (mindspore_amd/csrc/slot_pool.h, compiled for the host with sets that are no
memory): none before what the calls would have saved has come to a set's price, as many as callers at once up to a limit, all of
them given back with the last user."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <atomic>
#include <thread>
#include <vector>
#include "mindspore_amd/csrc/slot_pool.h"

static std::atomic<int> made{0}, live{0};
static bool no_memory = false;
struct Set {
  Set *next = nullptr;
  std::atomic<int> callers{0};
  static Set *make(int) {
    if (no_memory) return nullptr;
    ++made, ++live;
    return new Set();
  }
  static void free(Set *s) {
    --live;
    delete s;
  }
};
typedef mi::SlotPool<Set> Pool;
#define CHECK(c) if (!(c)) { printf("line %d: " #c " (made %d, live %d)\n", __LINE__, made.load(), live.load()); exit(1); }

static const size_t kBytes[2] = {256 << 10, 4 << 20};
static float saved(size_t bytes) { return 5.0f + 15.0f / (1 << 20) * (float)bytes; }
static bool pageable() { return true; }
static bool locked() { return false; }

int main() {
  Pool p;
  for (int size = 0; size < 2; ++size) {
    made = 0;
    // a handle per call
    for (int i = 0; i < 100; ++i) {
      p.add_user();
      Set *s = p.take(size, kBytes[size], pageable);
      CHECK(s == nullptr);
      p.drop_user();
    }
    CHECK(made == 0);
    // page-locked tensors
    p.add_user();
    for (int i = 0; i < 500; ++i) CHECK(p.take(size, kBytes[size], locked) == nullptr);
    p.drop_user();
    CHECK(made == 0);
    // one after the other: a single set, once it is worth it and not much later
    p.add_user();
    int first = -1;
    for (int i = 0; i < 200; ++i) {
      Set *s = p.take(size, kBytes[size], pageable);
      if (s != nullptr && first < 0) first = i;
      if (s != nullptr) p.give(size, s);
    }
    CHECK(made == 1 && live == 1);
    CHECK(first * saved(kBytes[size]) < Pool::kPrice && (first + 1) * saved(kBytes[size]) >= Pool::kPrice);
    // bursts of more callers than there may be sets: they stay from burst to burst, callers beyond go without
    for (int burst = 0; burst < 2000; ++burst) {
      std::vector<Set *> held;
      for (int c = 0; c < Pool::kMostSets + 4; ++c)
        if (Set *s = p.take(size, kBytes[size], pageable)) held.push_back(s);
      CHECK((int)held.size() <= Pool::kMostSets);
      if (burst > 1000) CHECK((int)held.size() == Pool::kMostSets);
      for (Set *s : held) p.give(size, s);
    }
    CHECK(made == Pool::kMostSets && live == Pool::kMostSets);
    // another user keeps them
    p.add_user();
    p.drop_user();
    CHECK(live == Pool::kMostSets);
    p.drop_user();
    CHECK(live == 0);
    // no page-locked memory: without, and a set as soon as there is some and it is worth it again
    p.add_user();
    no_memory = true;
    for (int i = 0; i < 200; ++i) CHECK(p.take(size, kBytes[size], pageable) == nullptr);
    no_memory = false;
    Set *s = nullptr;
    for (int i = 0; i < 200 && s == nullptr; ++i) s = p.take(size, kBytes[size], pageable);
    CHECK(s != nullptr);
    p.give(size, s);
    p.drop_user();
    CHECK(live == 0);
  }
  // threads that come and go
  std::atomic<int> served{0}, bad{0};
  std::vector<std::thread> threads;
  for (int t = 0; t < 12; ++t)
    threads.emplace_back([&, t] {
      for (int handle = 0; handle < 20; ++handle) {
        p.add_user();
        for (int call = 0; call < 300; ++call) {
          const int size = (call + t) & 1;
          Set *s = p.take(size, kBytes[size], pageable);
          if (s == nullptr) continue;
          if (s->callers.fetch_add(1) != 0) ++bad;
          ++served;
          s->callers.fetch_sub(1);
          p.give(size, s);
        }
        p.drop_user();
      }
    });
  for (std::thread &t : threads) t.join();
  CHECK(bad == 0 && served > 0 && live == 0);
  printf("ok\n");
  return 0;
}
"""


def test_sets_come_when_they_are_worth_it_and_go_with_the_last_user(tmp_path):
    src, exe = tmp_path / "pool.cc", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", "-I" + ROOT, str(src), "-o", str(exe)])
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and p.stdout == "ok\n", p.stdout
