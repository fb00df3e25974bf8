// gz_runtime.h -- the opaque stream handle of the C ABI, and the library's
// device memory calls.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

struct gz_stream_s {
  hipStream_t s;
};

struct gz_gapped_extender_s;

namespace gz {

// Whether a call of `size` jobs with the extender's present settings runs one
// wave per job (extenders.hip): the first ring's settings then change nothing.
bool GappedRunsRows(const gz_gapped_extender_s *h, size_t size);
// The extender's workspace for calls of up to `size` jobs with its present
// settings (gz_gapped_extender_reserve: with any); whether it could be had.
bool GappedReserveNow(gz_gapped_extender_s *h, size_t size, hipStream_t s);

// Stream capture and memory management exclude each other.  Freeing device
// or pinned memory synchronizes the device, which a capture in flight on
// another thread's stream forbids (the free fails with "operation not
// permitted when stream is capturing"); the library's captures and every
// allocation or free it makes mid-run hold this lock.
std::recursive_mutex &CaptureLock();

// Device workspaces of calls that keep none.  A call takes a
// block, is its only user until its kernels and copies have ended, and gives
// it back; one block per device is kept between calls, of at most kMost
// bytes, the largest given back (a call that finds none, or one too small,
// allocates its own; gz_release_workspaces frees them).  Mapping and unmapping a call's scratch costs far more
// than using it: 50,021 read results (140 MB of scratch) take 11 ms with an
// allocation per call and 1.34 ms without where other allocations of the
// process come and go, 3,001 protein results (300 MB) 12 and 0.67 ms.
class WorkspacePool {
 public:
  static constexpr size_t kMost = (size_t)512 << 20;
  // the current device's block: at least `bytes`, its size to *capacity
  static hipError_t Take(size_t bytes, void **p, size_t *capacity);
  // with the device current that the block was taken on and no work on the
  // block in flight
  static void Give(void *p, size_t capacity);
  // frees the kept blocks; whether there was one
  static bool Trim();
};

template <typename T>
inline hipError_t Malloc(T **p, size_t bytes) {
  std::lock_guard<std::recursive_mutex> g(CaptureLock());
  const hipError_t e = hipMalloc((void **)p, bytes);
  if (e != hipErrorOutOfMemory || !WorkspacePool::Trim()) return e;
  (void)hipGetLastError();
  return hipMalloc((void **)p, bytes);
}

template <typename T>
inline hipError_t HostMalloc(T **p, size_t bytes, unsigned flags = hipHostMallocDefault) {
  std::lock_guard<std::recursive_mutex> g(CaptureLock());
  return hipHostMalloc((void **)p, bytes, flags);
}

inline hipError_t Free(void *p) {
  std::lock_guard<std::recursive_mutex> g(CaptureLock());
  return hipFree(p);
}

inline hipError_t HostFree(void *p) {
  std::lock_guard<std::recursive_mutex> g(CaptureLock());
  return hipHostFree(p);
}

}  // namespace gz
