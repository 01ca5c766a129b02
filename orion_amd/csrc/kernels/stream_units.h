// Compute units that a stream may use.
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace stream_units {

constexpr int kWholeGpu = 256;

// Asks the stream for its mask (0.2 us); the whole GPU where that cannot be told.  The
// runtime's own streams (null, legacy, per thread) have none, and their handles are
// constants that only launches are sure to take.
inline int compute_units_of(hipStream_t stream) {
  if (stream == nullptr || stream == hipStreamLegacy || stream == hipStreamPerThread)
    return kWholeGpu;
  uint32_t mask[16] = {0};
  if (hipExtStreamGetCUMask(stream, 16, mask) != hipSuccess) {
    (void)hipGetLastError();
    return kWholeGpu;
  }
  int cus = 0;
  for (uint32_t word : mask) cus += __builtin_popcount(word);
  return cus > 0 && cus < kWholeGpu ? cus : kWholeGpu;
}

}  // namespace stream_units
