"""The timeline probes of profiling builds (VIB3_TRACE, csrc/common.h) on the CPU: a translation unit
whose buffer pointer nobody set must not store through it, a set one gets its value."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
COMMON = os.path.join(ROOT, "vib3_amd", "csrc", "common.h")

PROGRAM = r"""
#include <stdint.h>
#include <stdio.h>
#define VIB3_TRACE
#define __device__
#define __forceinline__ inline
static struct { unsigned x, y; } threadIdx, blockIdx;
static uint64_t __builtin_amdgcn_s_memrealtime() { return 42; }
%s
int main() {
  VIB3_TRACE_POINT(3);
  VIB3_TRACE_VALUE(4, 7);
  uint64_t buf[64] = {0};
  vib3_trace_buf = buf;
  blockIdx.x = 2;
  VIB3_TRACE_POINT(3);
  VIB3_TRACE_VALUE(4, 7);
  threadIdx.x = 1;
  VIB3_TRACE_VALUE(5, 9);
  return buf[35] == 42 && buf[36] == 7 && buf[37] == 0 ? 0 : 1;
}
"""


def test_probes_skip_an_unset_buffer(tmp_path):
    probes = re.search(r"^#ifdef VIB3_TRACE\n.*?^#endif\n", open(COMMON).read(), re.M | re.S).group(0)
    src, exe = tmp_path / "probes.cpp", tmp_path / "probes"
    src.write_text(PROGRAM % probes)
    subprocess.run(["g++", "-std=c++17", "-o", str(exe), str(src)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


def test_probe_buffer_is_written_in_one_place():
    """Every probe of the sources goes through the guarded store."""
    csrc = os.path.dirname(COMMON)
    stores = [(f, line) for f in sorted(os.listdir(csrc)) for line in open(os.path.join(csrc, f))
              if re.search(r"vib3_trace_buf\s*\[", line)]
    assert len(stores) == 1 and "if (threadIdx.x == 0 && vib3_trace_buf)" in stores[0][1], stores
