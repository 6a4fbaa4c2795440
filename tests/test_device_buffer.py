"""The owning device buffer (csrc/common.h) when an allocation fails, compiled for the CPU
against a stand-in for the allocator: it is empty then, so that a caller that checks its size
allocates again instead of handing a null pointer to a kernel."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "xrtailor_amd" / "csrc"

DRIVER = r"""
#include <cstdlib>
#include "common.h"
static bool fail = false;
static int live = 0;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (fail) {
    *p = reinterpret_cast<void*>(8);  // a failed call may leave anything there
    return hipErrorOutOfMemory;
  }
  *p = std::malloc(n);
  ++live;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::free(p);
  --live;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}
int main() {
  {
    xrt::DevBuf<int> b;
    if (b.Alloc(10) != hipSuccess || !b.ptr || b.n != 10) return 1;
    fail = true;
    if (b.Alloc(20) != hipErrorOutOfMemory || b.ptr || b.n != 0) return 2;
    if (b.Upload(std::vector<int>(20, 1), nullptr) != hipErrorOutOfMemory || b.ptr || b.n != 0) return 3;
    if (b.Alloc(0) != hipSuccess || b.ptr || b.n != 0) return 4;
    fail = false;
    if (b.Alloc(20) != hipSuccess || !b.ptr || b.n != 20) return 5;
  }
  return live == 0 ? 0 : 6;
}
"""


def test_failed_allocation_leaves_an_empty_buffer(tmp_path):
    (tmp_path / "main.cpp").write_text(DRIVER)
    exe = tmp_path / "buffer"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", str(tmp_path / "main.cpp"), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
