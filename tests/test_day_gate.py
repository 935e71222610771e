"""The gate before the many-days kernel (watergap2_amd/csrc/wg_day_gate.h), compiled for
the CPU: threads that enter with wavefront counts below, at and above the limit run
together only while the sum is within it, a larger one runs alone, all of them get their
turn, and in the order they came."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "watergap2_amd", "csrc")

SRC = r"""
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#include "wg_day_gate.h"

int main() {
  constexpr int64_t limit = 1024;
  const int64_t waves[] = {1, 32, 500, 512, 524, 1023, 1024, 1025, 1127, 36064};
  WgDayGate gate;
  std::atomic<int64_t> running{0}, calls{0}, most{0};
  std::atomic<int> inside{0}, bad{0}, together{0};
  std::vector<std::thread> threads;
  for (int t = 0; t < 8; t++)
    threads.emplace_back([&, t] {
      for (int i = 0; i < 400; i++) {
        const int64_t w = waves[(i * 7 + t * 3) % 10];
        gate.enter(w, limit);
        const int64_t sum = running += w;
        const int n = ++inside;
        if (n > 1 && sum > limit) bad++;
        if (n > 1) together++;
        std::this_thread::sleep_for(std::chrono::microseconds(5));
        inside--;
        running -= w;
        gate.leave(w);
        calls++;
      }
    });
  for (auto &t : threads) t.join();
  // turns: while one that fills the chip runs, a second and a third wait; the third is
  // small but does not pass the second
  std::atomic<int> order{0}, second{0}, third{0};
  gate.enter(2000, limit);
  std::thread b([&] { gate.enter(1500, limit); second = ++order; gate.leave(1500); });
  std::this_thread::sleep_for(std::chrono::milliseconds(50));
  std::thread c([&] { gate.enter(1, limit); third = ++order; gate.leave(1); });
  std::this_thread::sleep_for(std::chrono::milliseconds(50));
  const int early = order;
  gate.leave(2000);
  b.join();
  c.join();
  std::printf("%ld %d %d %d %d %d\n", long(calls), int(bad), int(together), early, int(second), int(third));
}
"""


def test_gate_keeps_launches_apart_that_do_not_fit(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    src, exe = str(tmp_path / "gate.cpp"), str(tmp_path / "gate")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-pthread", "-I", CSRC, src, "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout
    calls, bad, together, early, second, third = map(int, out.split())
    assert calls == 3200 and bad == 0 and together > 0
    assert early == 0 and (second, third) == (1, 2)
