"""Host-only: what the launchers set once per GPU (a kernel's LDS limit) is set on
every device, by whichever thread comes first, and tried again after a failure."""
import os
import subprocess

from fft_amd import build as B

SRC = r"""
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
#include "afft_per_device.h"

int main() {
  afgpu::PerDevice d;
  std::atomic<int> calls[3] = {};
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 12; t++)
    ts.emplace_back([&, t] {
      for (int i = 0; i < 1000; i++) {
        const int dev = (t + i) % 3;
        if (d.once(dev, [&] { calls[dev]++; return 0; }) != 0 || calls[dev] == 0) bad++;
      }
    });
  for (auto& t : ts) t.join();
  for (int dev = 0; dev < 3; dev++)
    if (calls[dev] < 1 || calls[dev] > 12) bad++;
  afgpu::PerDevice f;
  if (f.once(5, [] { return 7; }) != 7 || f.once(5, [] { return 0; }) != 0 || f.once(5, [] { return 7; }) != 0) bad++;
  // a device number past the flags is set each time
  if (f.once(64, [] { return 0; }) != 0 || f.once(64, [] { return 3; }) != 3) bad++;
  printf("%d\n", bad.load());
  return bad.load() != 0;
}
"""


def test_once_per_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", B.CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


def test_no_launcher_keeps_a_process_wide_flag():
    for f in sorted(os.listdir(B.CSRC)):
        assert "static bool attr" not in open(os.path.join(B.CSRC, f)).read(), f
