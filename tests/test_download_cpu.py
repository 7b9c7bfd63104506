"""Host side of the downloads (csrc/ek_hostcopy.h) with the device copy replaced by a stub: a copy
that fails leaves the destination as it was, whether its pages are in memory or not, and one that
succeeds fills it (FP32 widened), at sizes of one part, of two and of the most. A destination that
is device memory is the copy's alone to write."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "euler_kokkos_amd", "csrc")
ROCM = "/opt/rocm/include"

DRIVER = r"""
#include "ek_hostcopy.h"
#include <cstdio>
#include <cstring>
#include <vector>
#include <sys/mman.h>

static bool fails;
static const void* device; // stands for device memory: no access from the host
extern "C" hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t)
{
  if (fails)
    return hipErrorUnknown;
  memcpy(dst, src, n);
  return hipSuccess;
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
  a->type = hipMemoryTypeDevice;
  return p == device ? hipSuccess : hipErrorInvalidValue;
}
extern "C" hipError_t hipGetLastError() { return hipErrorInvalidValue; }

int main()
{
  int bad = 0;
  for (long long n : { 1000LL, 131072LL, 1048576LL + 3, 1179648LL, 8388608LL + 1 })
    for (int fp32 = 0; fp32 < 2; fp32++)
      for (int touched = 0; touched < 3; touched++) { // none, the first half, all of the destination
        std::vector<double> s64(n);
        std::vector<float> s32(n);
        for (long long i = 0; i < n; i++)
          s64[i] = s32[i] = (float)(i % 1237) + 0.5f;
        const void* src = fp32 ? (const void*)s32.data() : (const void*)s64.data();
        double* host = (double*)mmap(nullptr, n * 8, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        const size_t old = n * 8 / 2 * touched;
        memset((void*)host, 0xa5, old);
        fails = true;
        const bool err = ek::copy_to_host(host, src, fp32, n, nullptr) != hipSuccess;
        long long changed = 0;
        for (size_t i = 0; i < (size_t)n * 8; i++)
          changed += ((unsigned char*)host)[i] != (i < old ? 0xa5 : 0);
        fails = false;
        const bool ok = ek::copy_to_host(host, src, fp32, n, nullptr) == hipSuccess;
        const bool same = memcmp(host, s64.data(), n * 8) == 0;
        if (!err || changed || !ok || !same) {
          printf("n %lld fp32 %d touched %d: failed copy reported %d, bytes it changed %lld; copy ok %d, right %d\n", n, fp32,
                 touched, err, changed, ok, same);
          bad++;
        }
        munmap(host, n * 8);
      }
  for (long long n : { 1000LL, 8388608LL + 1 }) {
    std::vector<double> s64(n);
    device = mmap(nullptr, n * 8, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    fails = true; // the stub has no way to write there either
    bad += ek::copy_to_host((double*)device, s64.data(), false, n, nullptr) == hipSuccess;
  }
  printf("%d bad\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(os.path.join(ROCM, "hip", "hip_runtime.h")) or not shutil.which("g++"),
                    reason="needs g++ and the HIP headers")
def test_copies_that_fail_and_that_succeed(tmp_path):
    src = tmp_path / "driver.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "driver"
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", ROCM, "-I", CSRC, str(src), "-o", str(exe),
                    "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
