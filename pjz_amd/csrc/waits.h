// Waits between the workgroups of one launch, bounded by the device's clock.
#pragma once

#include <hip/hip_runtime.h>

namespace pjz {

// Whether a stream's kernels may use all `cus` compute units of its device: a
// stream can be created with a mask, and workgroups that need them all at the
// same time have to keep off its others.
inline bool whole_device(hipStream_t s, int cus) {
  uint32_t mask[32] = {};
  if (cus > 32 * 32) return true;
  if (hipExtStreamGetCUMask(s, (cus + 31) / 32, mask) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  int n = 0;
  for (uint32_t m : mask) n += __builtin_popcount(m);
  return n == 0 || n >= cus;
}

// Workgroups that exchange words wait for one another.  Such a wait ends by
// itself where all of them are on the chip at the same time and nobody else
// writes the words.  A cooperative launch arranges the first on a GPU of its
// own only (another process may hold compute units), and the second is the
// callers' (overlapping calls must not share a workspace).  Where either
// fails, the launch's waits end after a time, its results are spoiled with
// NaN, and the host is told: no workgroup stays on the GPU for good.
//
// The time is counted in the device's clock, not in polls: kernels of other
// streams may hold back some of the workgroups for long.  A wave keeps its
// waits' end in LDS and looks at it and at the clock after kWaitPolls polls of
// a wait only: most waits end within a few polls, and a look at each made the
// smallest runs 3% slower.
struct WaitArgs {
  unsigned ticks;     // from a wave's start, kWaitTick of the clock's each
  unsigned* stalled;  // device word, set by waves that waited in vain: later
                      // launches that share it do not wait as long again
  unsigned* report;   // the same for the host
};
constexpr int kWaitTick = 1024;  // 10 us at 100 MHz; 32 bits last 6 hours
constexpr int kWaitPolls = 64;
constexpr unsigned kLate = 0;    // a wave's end of waits once one was in vain

__device__ __forceinline__ unsigned wait_clock() {
  return (unsigned)((unsigned long long)wall_clock64() / kWaitTick);
}
// The end of the waits of a wave that starts now.
__device__ __forceinline__ unsigned wait_end(const WaitArgs& a) {
  if (__hip_atomic_load(a.stalled, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return kLate;
  return (wait_clock() + a.ticks) | 1;
}
// Whether waits that end at `*end` are over, noted there.
__device__ __forceinline__ bool wait_over(unsigned* end) {
  const unsigned u = __builtin_amdgcn_readfirstlane(*end);
  if (u != kLate && (int)(wait_clock() - u) < 0) return false;
  *end = kLate;
  return true;
}
// Of a wave that waited in vain, at its end.
__device__ __forceinline__ void tell_late(const WaitArgs& a) {
  __hip_atomic_store(a.stalled, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(a.report, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace pjz
