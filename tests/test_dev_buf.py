"""The device buffer's bookkeeping, compiled for the host with stand-ins for the
allocation functions."""

import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <cstddef>
#include <cstdlib>
#include <stdexcept>
static int live = 0;
static bool fail = false;
static int hipMalloc(void** p, std::size_t n) {
  if (fail) return 2;
  *p = std::malloc(n);
  ++live;
  return 0;
}
static int hipMemset(void*, int, std::size_t) { return 0; }
static int hipFree(void* p) {
  std::free(p);
  --live;
  return 0;
}
#define XFD_HIP(x) do { if ((x) != 0) throw std::runtime_error(#x); } while (0)
#include "dev_buf.hpp"
int main() {
  {
    DevBuf b;
    b.alloc(100);
    if (!b.p || b.bytes != 100) return 1;
    fail = true;
    bool thrown = false;
    try { b.alloc(1000); } catch (const std::runtime_error&) { thrown = true; }
    if (!thrown || b.p || b.bytes != 0) return 2;  // holds nothing and says so
    fail = false;
    b.alloc(500);
    if (!b.p || b.bytes != 500) return 3;
    DevBuf c = static_cast<DevBuf&&>(b);
    if (b.p || b.bytes || c.bytes != 500) return 4;
  }
  return live == 0 ? 0 : 5;
}
"""


def test_a_failed_allocation_holds_nothing(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", f"-I{ROOT / 'xfdtd_core_amd' / 'csrc' / 'device'}", str(src), "-o", str(exe)],
                   check=True)
    assert subprocess.run([str(exe)]).returncode == 0
