// traceback.h -- the result build's traceback re-extensions on the device.
#pragma once

#include <stdint.h>

#include <hip/hip_runtime.h>

#include "presearch.h"

namespace gz {

// Per-lane scratch capacities (elements) and the lane stride in bytes.
struct LaneCaps {
  uint32_t dp = 0, rows = 0, arena = 0, ops = 0;
  size_t bytes_per_lane = 0;
};

// The op arena of a side, in bytes; a side whose rows need more is flagged.
constexpr uint32_t kTracebackArena = 1u << 16;

// Packed sequences, score parameters and the bounds of the jobs: the longest
// framed query, the longest subject.
struct TracebackInputs {
  const uint64_t *queries, *database;
  uint32_t max_query_length, max_subject_length;
  uint32_t longest_side;  // residues between two of a query's delimiters, at most
  const int *matrix;  // on the device
  uint32_t nl;
  int gap_open, gap_ext, cutoff;
};

// Runs jobs, one after the other call, in a workspace that it keeps (pooled:
// that it takes from the library's pool and gives back at its end).
class TracebackRunner {
 public:
  explicit TracebackRunner(bool pooled = false) : pooled_(pooled) {}
  ~TracebackRunner();
  TracebackRunner(const TracebackRunner &) = delete;
  TracebackRunner &operator=(const TracebackRunner &) = delete;
  // jobs and outs on the host; synchronous.  kernel_ms (may be null): the
  // kernels' time.
  hipError_t Run(const TracebackInputs &in, const TracebackJob *jobs, uint32_t n,
                 TracebackOut *outs, hipStream_t s, float *kernel_ms);

 private:
  hipError_t Queue(const TracebackInputs &in, const TracebackJob *jobs, uint32_t n,
                   TracebackOut *outs, hipStream_t s, float *kernel_ms);
  hipError_t Reserve(size_t bytes, void **p, size_t *capacity);
  void Release(void **p, size_t *capacity);
  // `before` bytes and the lanes' scratch, for fewer lanes while memory lacks
  hipError_t ReserveLanes(size_t before, size_t lanes, size_t bytes_per_lane, void **p,
                          size_t *capacity);
  // one lane per job (d_list: the n jobs to run), as many as `bytes` of scratch hold
  hipError_t Lanes(const TracebackInputs &in, const TracebackJob *d_jobs, uint32_t n,
                   const uint32_t *d_list, TracebackOut *d_outs, uint8_t *scratch, size_t bytes,
                   hipStream_t s);
  const bool pooled_;
  void *ws_ = nullptr, *lane_ws_ = nullptr;
  size_t cap_ = 0, lane_cap_ = 0;
  hipEvent_t ev_[2] = {nullptr, nullptr};
};

}  // namespace gz
