"""The reservation of resident blocks (glx_slots.h) in host threads: within
the cap, and in the order asked for, so that a large solve gets its turn while
small ones, which would fit beside each other, keep coming; and launches that
fit the device together fit each of its XCDs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#include "glx_slots.h"
using glx::FairSlots;

static int fail(const char* what) {
  std::printf("%s\n", what);
  return 1;
}
static void until_waiting(FairSlots& s, int n) {
  for (int k = 0; k < 2000 && s.waiting() < n; k++) std::this_thread::sleep_for(std::chrono::milliseconds(1));
}

int main() {
  const int cap = 10;
  {
    // 4 in use; 8 have to wait, and a later 4 that would fit waits behind them
    FairSlots s;
    std::atomic<int> order{0}, big{0}, small{0};
    s.acquire(4, cap);
    std::thread b([&] { s.acquire(8, cap); big = ++order; s.release(8); });
    until_waiting(s, 1);
    std::thread c([&] { s.acquire(4, cap); small = ++order; s.release(4); });
    until_waiting(s, 2);
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    const bool passed = small != 0 || s.used() != 4;
    s.release(4);
    b.join();
    c.join();
    if (passed) return fail("a later caller was served first");
    if (big != 1 || small != 2 || s.used() != 0) return fail("wrong order");
  }
  {
    // more than the cap: alone, rather than never
    FairSlots s;
    s.acquire(cap + 2, cap);
    s.release(cap + 2);
  }
  {
    // many threads of several sizes: never beyond the cap, every one served
    FairSlots s;
    std::atomic<int> used{0}, over{0}, served{0};
    std::vector<std::thread> ts;
    for (int t = 0; t < 8; t++)
      ts.emplace_back([&, t] {
        const int n = 1 + t;
        for (int k = 0; k < 500; k++) {
          s.acquire(n, cap);
          if ((used += n) > cap) over++;
          used -= n;
          s.release(n);
          served++;
        }
      });
    for (auto& t : ts) t.join();
    if (over != 0) return fail("beyond the cap");
    if (served != 4000 || s.used() != 0 || s.waiting() != 0) return fail("not everyone was served");
  }
  {
    // two launches within 256 CUs, and three: each XCD's share within its 32
    auto share = [](int blocks) { return (blocks + 7) / 8; };
    for (int a = 1; a <= 256; a++)
      for (int b = 1; b <= a; b++) {
        const int two = glx::resident_slots(a) + glx::resident_slots(b);
        if (two <= 256 && share(a) + share(b) > 32) return fail("two launches beyond an XCD");
        for (int c = 1; c <= b; c++)
          if (two + glx::resident_slots(c) <= 256 && share(a) + share(b) + share(c) > 32)
            return fail("three launches beyond an XCD");
      }
    if (glx::resident_slots(256) != 256 || glx::resident_slots(1) > 256) return fail("a launch that no longer fits");
  }
  std::printf("ok\n");
  return 0;
}
"""


def test_reservation(tmp_path):
    src, exe = tmp_path / "slots.cpp", tmp_path / "slots"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "generic-linalg_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
