// ftm_once.h -- a call that has to be made once per device (host code, no HIP
// headers: the CPU test compiles it by itself).
#pragma once

#include <atomic>
#include <cstdint>

namespace ftm {

// Whether something was done on each device of the process: a bit a device,
// set only after it succeeded.  Two threads may both do it; that must be
// harmless.
using DeviceBits = std::atomic<uint64_t>;

// set() (0 = success) unless it has succeeded on device `dev` before; devices
// from 64 on are set every time.
template <class Set>
inline int once_per_device(DeviceBits& done, int dev, Set&& set) {
  const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t{1} << dev : 0;
  if (bit != 0 && (done.load(std::memory_order_acquire) & bit) != 0) return 0;
  const int rc = set();
  if (rc == 0 && bit != 0) done.fetch_or(bit, std::memory_order_release);
  return rc;
}

}  // namespace ftm
