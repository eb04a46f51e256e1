"""The per-device launch-size cache (csrc/device_cache.h) read by several host threads at once, under
the thread sanitizer. Launches take no lock around it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <thread>
#include <vector>
#include "device_cache.h"
static int grid(int dev) {
  static vib3::DeviceCache cache;
  return cache.get(dev, [&] { return 100 + dev; });
}
int main() {
  int bad[8] = {0};
  std::vector<std::thread> t;
  for (int i = 0; i < 8; i++)
    t.emplace_back([i, &bad] {
      for (int n = 0; n < 1000; n++)
        for (int dev = 0; dev < 4; dev++) bad[i] += grid(dev) != 100 + dev;
    });
  for (auto& x : t) x.join();
  int sum = 0;
  for (int b : bad) sum += b;
  return sum;
}
"""


def test_cache_has_no_data_race(tmp_path):
    src, exe = tmp_path / "cache.cpp", tmp_path / "cache"
    src.write_text(PROGRAM)
    built = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=thread", "-I",
                            os.path.join(ROOT, "vib3_amd", "csrc"), "-o", str(exe), str(src)],
                           capture_output=True, text=True)
    if built.returncode != 0 and "tsan" in built.stderr:
        pytest.skip("no thread sanitizer runtime")
    assert built.returncode == 0, built.stderr
    ran = subprocess.run([str(exe)], capture_output=True, text=True)
    if "unexpected memory mapping" in ran.stderr:
        pytest.skip("the thread sanitizer does not run on this kernel")
    assert ran.returncode == 0, ran.stderr


def test_launchers_keep_no_other_cache():
    """No launcher keeps a plain static int of its own (the streams and events of the MXFP4 batches
    are created and used under a lock)."""
    csrc = os.path.join(ROOT, "vib3_amd", "csrc")
    for name in sorted(os.listdir(csrc)):
        for line in open(os.path.join(csrc, name)):
            assert not line.lstrip().startswith(("static int grid", "static int cus")), (name, line)
