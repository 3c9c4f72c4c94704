"""CPU: a plan's device buffer (wh_devbuf.hpp) after an allocation that fails.  Plans compare its
size with what a call needs (moments of the adjoint steps, coefficient rows) and launch kernels on
its address: after a failure both must be those of the allocation that is there.  The header is
compiled for the host with an allocator of its own that can be told to fail."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "pywignercuda_amd" / "csrc"

PROGRAM = r"""
#include "wh_devbuf.hpp"
#include <cstdio>
#include <cstdlib>
static bool failing = false;
static int live = 0;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
  if (failing) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  ++live;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
  std::free(p);
  --live;
  return hipSuccess;
}
int main() {
  {
    wh::DeviceBuffer b;
    failing = true;
    if (b.replace(64) != hipErrorOutOfMemory || b.p || b.bytes) return std::puts("first failure"), 1;
    failing = false;
    if (b.replace(64) != hipSuccess || !b.p || b.bytes != 64) return std::puts("first allocation"), 1;
    void* const old = b.p;
    failing = true;
    if (b.replace(1 << 20) != hipErrorOutOfMemory || b.p != old || b.bytes != 64 || live != 1)
      return std::puts("failure of a larger one"), 1;
    failing = false;
    if (b.replace(1 << 20) != hipSuccess || b.bytes != (1 << 20) || live != 1) return std::puts("growth"), 1;
  }
  if (live) return std::puts("leak"), 1;
  return 0;
}
"""


def test_buffer_keeps_its_allocation_when_a_new_one_fails(tmp_path):
    cxx, hip = shutil.which("g++"), Path("/opt/rocm/include/hip/hip_runtime_api.h")
    if cxx is None or not hip.exists():
        pytest.skip("needs g++ and the HIP headers")
    src, exe = tmp_path / "buffer.cpp", tmp_path / "buffer"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}", str(src), "-o",
                    str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
