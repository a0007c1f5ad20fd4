// Large results to the caller's pageable memory.
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>

#include "ptyk_internal.h"

namespace ptyk {

// A result array is usually fresh, so the copy out also pays for its pages: hipMemcpyAsync takes them
// one by one and copies in one thread (52 MB: 5.0 ms; into pages that are there 2.9; to pinned memory
// 0.93).  Here a few threads move pieces through pinned buffers, two each, so that the pages, the copies
// and the transfers overlap.  Pieces are huge pages of dst: two threads that meet in one would both clear
// it.  52 MB with its simulation: 6.0 -> 2.2 ms; 8 threads instead of 4 the same, pieces of 1 MiB 2.5 and
// of 512 KiB 3.3 ms.  4 MB with theirs: 0.51 -> 0.43 ms.  Below HC_MIN the threads and buffers cost what
// they save.
static constexpr size_t HC_PIECE = 2 << 20;
static constexpr int HC_THREADS = 4;
static constexpr size_t HC_MIN = 4 << 20;

namespace {
struct Job {
  char* dst;
  const char* src;
  size_t bytes;
  int device;
  hipStream_t s;
  const hipEvent_t* ready;
  size_t per_event;
  char* pinned;  // two pieces per worker
  std::atomic<size_t> next{0};
  std::atomic<int> err{0};

  hipError_t work(int t) {
    hipError_t e = hipSetDevice(device);
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (auto& x : ev)
      if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    size_t at[2], len[2] = {0, 0};
    for (int b = 0; e == hipSuccess; b ^= 1) {
      char* buf = pinned + (size_t)(2 * t + b) * HC_PIECE;
      // the first piece ends where dst's first huge page does
      const size_t p = next.fetch_add(1), skip = (uintptr_t)dst % HC_PIECE;
      at[b] = p ? p * HC_PIECE - skip : 0;
      len[b] = at[b] < bytes ? std::min(p ? HC_PIECE : HC_PIECE - skip, bytes - at[b]) : 0;
      if (len[b]) {
        // the pieces come in order, so waiting for the event of a piece's last byte covers all of it
        if (ready) e = hipStreamWaitEvent(s, ready[(at[b] + len[b] - 1) / per_event], 0);
        if (e == hipSuccess) e = hipMemcpyAsync(buf, src + at[b], len[b], hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev[b], s);
      }
      const int o = b ^ 1;
      if (e == hipSuccess && len[o]) {
        e = hipEventSynchronize(ev[o]);
        if (e == hipSuccess) memcpy(dst + at[o], pinned + (size_t)(2 * t + o) * HC_PIECE, len[o]);
        len[o] = 0;
      }
      if (!len[b]) break;
    }
    for (auto x : ev)
      if (x) hipEventDestroy(x);
    if (e != hipSuccess) {
      err.store((int)e);
      next.store(bytes / HC_PIECE + 2);  // the other workers finish what they have begun
    }
    return e;
  }
};
}  // namespace

hipError_t copy_to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t s, const hipEvent_t* ready,
                        size_t per_event) {
  const int cpus = (int)std::thread::hardware_concurrency();
  const int nt = std::min(HC_THREADS, cpus > 0 ? cpus : 1);
  Job j;
  if (bytes < HC_MIN || nt < 2 ||
      hipHostMalloc((void**)&j.pinned, (size_t)nt * 2 * HC_PIECE, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();  // no pinned memory to be had: the plain copy needs none
    hipError_t e = hipSuccess;
    if (ready && bytes) e = hipStreamWaitEvent(s, ready[(bytes - 1) / per_event], 0);
    if (e == hipSuccess) e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
  }
  j.dst = (char*)dst;
  j.src = (const char*)src;
  j.bytes = bytes;
  j.device = device;
  j.s = s;
  j.ready = ready;
  j.per_event = per_event;
  std::thread th[HC_THREADS];
  for (int t = 1; t < nt; ++t) {
    try {
      th[t] = std::thread([&j, t] { j.work(t); });
    } catch (...) {  // no more threads: those that run share the pieces
      break;
    }
  }
  j.work(0);
  for (auto& t : th)
    if (t.joinable()) t.join();
  hipError_t e = hipStreamSynchronize(s);
  hipHostFree(j.pinned);
  return j.err.load() ? (hipError_t)j.err.load() : e;
}

}  // namespace ptyk
