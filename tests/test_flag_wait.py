"""How the host waits for copies that run beside one another (mindspore_amd/csrc/flag_wait.h, compiled for the host with a stream that is no
stream): one that says idle once the last copy is over is not taken to have lost an earlier one, and a copy without its result, or a
stream that fails, ends the wait."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <atomic>
#include <thread>
#include "mindspore_amd/csrc/flag_wait.h"

// Three parts of one copy: two come with the drain, when the stream has long said idle.
struct Beside {
  uint32_t flags[3] = {7, 6, 6};
  int asked = 0, drained = 0, busy = 0, fails = 0, drain_fails = 0;
  bool lost = false;
  int idle(bool *idle) {
    *idle = ++asked > busy;
    return fails;
  }
  int drain() {
    ++drained;
    if (!lost) flags[1] = flags[2] = 7;
    return drain_fails;
  }
  int wait() { return mi::await_flags(flags, 3, 7, *this); }
};

static void check(bool good, const char *what) {
  if (good) return;
  printf("%s\n", what);
  exit(1);
}

int main() {
  Beside early;
  check(early.wait() == 0 && early.drained == 1, "idle by the last copy alone: the earlier one's flags come with the drain");
  Beside busy;
  busy.busy = 3;
  check(busy.wait() == 0 && busy.asked == 4, "asked again while the stream is busy");
  Beside lost;
  lost.lost = true;
  check(lost.wait() == mi::kFlagMissing && lost.drained == 1, "a copy without its result");
  lost.flags[1] = 7;  // (the last part alone)
  check(lost.wait() == mi::kFlagMissing, "a part without its result");
  Beside broken;
  broken.fails = -1;
  check(broken.wait() == -1 && broken.drained == 0, "a stream that fails");
  Beside late;
  late.drain_fails = -1;
  check(late.wait() == -1, "a stream that fails while it is waited for");
  Beside there;
  there.flags[1] = there.flags[2] = 7;
  check(there.wait() == 0 && there.asked == 0, "flags that are there: nothing is asked");
  Beside other;
  other.busy = 1 << 30;
  std::thread copy([&] {
    for (int w = 1; w < 3; ++w) __atomic_store_n(other.flags + w, 7u, __ATOMIC_RELEASE);
  });
  check(other.wait() == 0 && other.drained == 0, "flags that come while the stream is busy");
  copy.join();
  printf("ok\n");
  return 0;
}
"""


def test_copies_beside_one_another_are_waited_for(tmp_path):
    src, exe = tmp_path / "flags.cc", tmp_path / "flags"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", "-I" + ROOT, str(src), "-o", str(exe)])
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
