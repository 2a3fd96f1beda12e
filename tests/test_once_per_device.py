"""Host code that allows a kernel its dynamic LDS (csrc/ftm_once.h): once on
each device of the process, again after a failure, from several threads
without a data race (g++, ThreadSanitizer on this host code alone)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "freetoken-intel_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "ftm_once.h"
#define CHECK(c) if (!(c)) { std::printf("failed: %s\n", #c); return 1; }
int main() {
  static ftm::DeviceBits done;
  int calls = 0;
  auto ok = [&] { ++calls; return 0; };
  auto bad = [&] { ++calls; return 7; };
  CHECK(ftm::once_per_device(done, 0, bad) == 7 && calls == 1);  // a failure is not kept
  CHECK(ftm::once_per_device(done, 0, ok) == 0 && calls == 2);
  CHECK(ftm::once_per_device(done, 0, bad) == 0 && calls == 2);
  CHECK(ftm::once_per_device(done, 1, ok) == 0 && calls == 3);   // the next device needs its own
  CHECK(ftm::once_per_device(done, 63, ok) == 0 && calls == 4);
  for (int i = 0; i < 3; ++i) CHECK(ftm::once_per_device(done, 64 + i % 2, ok) == 0 && calls == 5 + i);
  static ftm::DeviceBits shared;
  std::atomic<int> sets{0};
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([&, t] {
      for (int i = 0; i < 1000; ++i) ftm::once_per_device(shared, (t + i) % 8, [&] { ++sets; return 0; });
    });
  for (auto& t : th) t.join();
  CHECK(sets >= 8 && sets <= 64);
  std::puts("once_per_device: ok");
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_once_per_device(tmp_path):
    src, exe = tmp_path / "once.cpp", str(tmp_path / "once")
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=thread", "-static-libtsan", "-I", CSRC,
                    str(src), "-o", exe], check=True, capture_output=True, text=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "once_per_device: ok" in r.stdout, r.stdout + r.stderr[-4000:]
