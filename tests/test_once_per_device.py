"""``csrc/once_per_device.h``: the opt-in of a kernel is made once for every device, not once for the process (CPU only)."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "once_per_device.h"
#include <cstdio>
#include <thread>
#include <vector>
int main() {
  static sjhip::OncePerDevice once;
  static std::atomic<int> made[3];
  std::vector<std::thread> threads;
  for (int i = 0; i < 16; ++i)
    threads.emplace_back([i]() { for (int n = 0; n < 1000; ++n) once(i % 2, [&]() { ++made[i % 2]; return 0; }); });
  for (auto &t : threads) t.join();
  int failed = 0;
  for (int n = 0; n < 3; ++n) failed += once(2, [&]() { ++made[2]; return n < 2 ? 7 : 0; });
  const int after = once(2, [&]() { ++made[2]; return 7; }), outside = once(-1, []() { return 5; });
  std::printf("%d %d %d %d %d %d\n", made[0].load(), made[1].load(), made[2].load(), failed, after, outside);
}
"""


def test_every_device_is_served_once_and_a_failure_is_tried_again(tmp_path):
    source, program = tmp_path / "once.cpp", tmp_path / "once"
    source.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "spikingjelly_amd", "csrc"), str(source), "-o", str(program)])
    # both devices once, however many threads ask; two failures (7 each), then done; no device: asked every time
    assert subprocess.check_output([str(program)], text=True).split() == ["1", "1", "3", "14", "0", "5"]
