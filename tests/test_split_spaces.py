"""Whose the memory is through which split GEMMs on the library's streams hand over their sums (mindspore_amd/csrc/split_spaces.h,
compiled for the host with spaces that are no memory): one for each stream from its creation to its end, never two streams' at
once, never the next stream's before the last one's work is done with it, none given back while there are streams, all with the
last."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <atomic>
#include <map>
#include <set>
#include <thread>
#include <vector>
#include "mindspore_amd/csrc/split_spaces.h"

static std::mutex m;
static std::map<void *, int> made;  // -> the stream that it was made for
static bool no_memory = false, held_up = false;
struct Fake {
  typedef int Stream;
  static void *make(int stream) {
    std::lock_guard<std::mutex> lock(m);
    if (no_memory) return nullptr;
    void *p = malloc(1);
    made[p] = stream;
    return p;
  }
  static bool free(void *p) {
    std::lock_guard<std::mutex> lock(m);
    if (held_up) return false;
    if (made.erase(p) != 1) { printf("freed what was not made\n"); exit(1); }
    ::free(p);
    return true;
  }
};
typedef mi::SplitSpaces<Fake> Spaces;
#define CHECK(c) if (!(c)) { printf("line %d: " #c " (%d made)\n", __LINE__, (int)made.size()); exit(1); }
static char there[2][3];  // for good, on devices 0 and 1

static void fill(Spaces &s) {
  for (int d = 0; d < 2; ++d)
    for (char &c : there[d]) s.keep(d, &c);
}
static void end(Spaces &s, int stream, bool destroyed = true, bool settled = true) { s.left(s.leave(stream), destroyed, settled); }

int main() {
  Spaces s;
  fill(s);
  CHECK(s.of(1) == nullptr && s.leave(1) == nullptr);
  s.left(nullptr, true, true);
  // the ones that are there first, on the stream's device; then ones that are made
  std::set<void *> seen;
  for (int i = 1; i <= 5; ++i) {
    s.enter(i, 0);
    void *p = s.of(i);
    CHECK(p != nullptr && seen.insert(p).second);
    CHECK((made.count(p) == 1) == (i > 3) && (i > 3 || ((char *)p >= there[0] && (char *)p < there[0] + 3)));
  }
  s.enter(6, 1);
  CHECK((char *)s.of(6) >= there[1] && (char *)s.of(6) < there[1] + 3);
  // one that was there is the next stream's once its stream's work is done
  void *of2 = s.of(2), *p = s.leave(2);
  CHECK(p == of2 && s.of(2) == nullptr);
  s.enter(7, 0);
  CHECK(s.of(7) != of2 && made.count(s.of(7)) == 1);
  s.left(p, true, true);
  s.enter(8, 0);
  CHECK(s.of(8) == of2);
  // and nobody's if that is not known
  end(s, 8, true, false);
  s.enter(9, 0);
  CHECK(s.of(9) != of2 && made.count(s.of(9)) == 1);
  // a stream that could not be destroyed keeps its space
  void *of3 = s.of(3), *of9 = s.of(9);
  end(s, 3, false, true);
  end(s, 9, false, false);
  CHECK(s.of(3) == of3 && s.of(9) == of9);
  // no memory: without
  no_memory = true;
  s.enter(10, 0);
  CHECK(s.of(10) == nullptr && s.leave(10) == nullptr);
  no_memory = false;
  // a made one stays for the next stream on its device, and is not given back before the last one's end
  void *of4 = s.of(4);
  const int so_far = (int)made.size();
  end(s, 4);
  CHECK((int)made.size() == so_far);
  s.enter(11, 1), s.enter(12, 1), s.enter(13, 1);
  CHECK((int)made.size() == so_far + 1);
  s.enter(14, 0);
  CHECK(s.of(14) == of4 && (int)made.size() == so_far + 1);
  end(s, 14, true, false);  // (nobody's, but given back with the others)
  for (int i : {1, 3, 5, 6, 7, 9, 11, 12}) {
    end(s, i);
    CHECK((int)made.size() == so_far + 1);
  }
  // if it cannot be given back then: with the next last one
  held_up = true;
  end(s, 13);
  CHECK((int)made.size() == so_far + 1);
  held_up = false;
  s.enter(15, 1);
  CHECK((int)made.size() == so_far + 1);
  end(s, 15);
  CHECK(made.empty());
  // one session after the other costs nothing
  for (int i = 100; i < 200; ++i) {
    s.enter(i, 0);
    CHECK(s.of(i) != nullptr && made.empty());
    end(s, i);
  }
  // many threads, each with streams of its own: a space is one stream's at a time
  Spaces t;
  fill(t);
  static std::atomic<int> owner[6];
  std::vector<std::thread> threads;
  for (int k = 0; k < 8; ++k)
    threads.emplace_back([&t, k] {
      for (int i = 0; i < 2000; ++i) {
        const int stream = 1 + 8 * i + k;
        t.enter(stream, k & 1);
        char *q = (char *)t.of(stream);
        CHECK(q != nullptr);
        const bool kept = q >= there[0] && q < there[0] + 6;
        if (kept) {
          CHECK((q - there[0]) / 3 == (k & 1));
          CHECK(owner[q - there[0]].exchange(stream) == 0);
          CHECK(owner[q - there[0]].exchange(0) == stream);
        }
        end(t, stream);
      }
    });
  for (std::thread &th : threads) th.join();
  CHECK(made.empty());
  printf("ok\n");
}
"""


def test_split_spaces(tmp_path):
    source, program = tmp_path / "spaces.cc", tmp_path / "spaces"
    source.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I" + ROOT, str(source), "-o",
                           str(program)])
    out = subprocess.run([str(program)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
