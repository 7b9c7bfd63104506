// ek_hostcopy.h -- device state to caller's (pageable) host memory, as FP64.
//
// Half the time of a large copy into memory that is not touched yet goes into its page faults,
// taken by the one thread that copies; an FP32 state was also widened on that thread. A few threads
// take the faults first, and widen. Per download: 134 MB FP64 (128^3, 8 variables) 12.7 -> 9.0 ms,
// the same state from FP32 24 -> 10. (A ring of pinned slots with threads behind it took 6.0 ms for
// the first, but 31 on a context's first download, which pays for the ring.)
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <new>
#include <thread>

#include <sys/mman.h>

namespace ek {

// work(lo, hi) over parts of [0, n), by at most 8 threads with at least `grain` elements each
template <class F>
inline void in_parts(long long n, long long grain, F work)
{
  constexpr int MAX = 8;
  const int parts = (int)std::max(1LL, std::min<long long>(MAX, n / grain));
  std::thread th[MAX];
  int started = 1; // part 0 is done here
  try {
    for (; started < parts; started++)
      th[started] = std::thread(work, n * started / parts, n * (started + 1) / parts);
  } catch (...) { // no more threads to be had: the rest is done here
  }
  work(0, n / parts);
  if (started < parts)
    work(n * started / parts, n);
  for (int t = 1; t < started; t++)
    th[t].join();
}

// Whether there are page faults to be taken in [mem, mem + bytes): not in memory the runtime knows
// (pinned, or the device's: no page of the host's to touch), nor where a page at each eighth of it
// is in memory.
inline bool faults(const char* mem, long long bytes)
{
  hipPointerAttribute_t at;
  const hipError_t e = hipPointerGetAttributes(&at, mem);
  if (e == hipSuccess && at.type != hipMemoryTypeUnregistered)
    return false;
  if (e != hipSuccess)
    (void)hipGetLastError(); // memory that the runtime does not know
  for (int i = 0; i < 8; i++) {
    unsigned char in = 0;
    if (mincore((void*)((unsigned long long)(mem + bytes / 8 * i) & ~4095ull), 1, &in) != 0 || !(in & 1))
      return true;
  }
  return false;
}

// Takes the page faults of memory that is about to be overwritten, where there are any and more
// than one thread to take them (from 8 MiB). What is in it stays as it is, since the copy may still
// fail: exchanging a zero byte for a zero byte is a write to the page whatever the byte is.
// (Touched again all the same, memory that is there costs 20 % of a pinned 34 MB download, 0.60 ms,
// and 8 % of a pageable one, 1.88.)
inline void touch(void* mem, long long bytes)
{
  constexpr long long GRAIN = 4 << 20;
  char* m = (char*)mem;
  if (bytes < 2 * GRAIN || !faults(m, bytes))
    return;
  in_parts(bytes, GRAIN, [m](long long lo, long long hi) {
    for (long long i = lo; i < hi; i += 4096) {
      char zero = 0;
      __atomic_compare_exchange_n(m + i, &zero, (char)0, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED);
    }
  });
}

// n values at device address src (double, or float with fp32) to host; returns when host is
// complete
inline hipError_t copy_to_host(double* host, const void* src, bool fp32, long long n, hipStream_t s)
{
  std::unique_ptr<float[]> part(fp32 ? new (std::nothrow) float[(size_t)n] : nullptr);
  if (fp32 && !part)
    return hipErrorOutOfMemory;
  void* to = fp32 ? (void*)part.get() : (void*)host;
  const long long bytes = n * (fp32 ? 4 : 8);
  touch(to, bytes);
  hipError_t e = hipMemcpyAsync(to, src, (size_t)bytes, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess)
    e = hipStreamSynchronize(s);
  if (fp32 && e == hipSuccess) {
    const float* f = part.get();
    in_parts(n, 1 << 19, [f, host](long long lo, long long hi) {
      for (long long i = lo; i < hi; i++)
        host[i] = (double)f[i];
    });
  }
  return e;
}

} // namespace ek
