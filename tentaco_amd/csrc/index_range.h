// Index arithmetic that holds up to the top of the int32 range, which a CSF's
// arrays may reach. Host and device, no HIP types, so that the CPU tests
// compile it alone.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define TT_HOST_DEVICE __host__ __device__ inline
#else
#define TT_HOST_DEVICE inline
#endif

namespace tt {

// min(at + ahead, last) for at, ahead and last in 0 .. 2^31-1, whose sum may
// pass 2^31-1.
TT_HOST_DEVICE int32_t index_ahead(int32_t at, int32_t ahead, int32_t last) {
  const uint32_t x = uint32_t(at) + uint32_t(ahead);
  return int32_t(x < uint32_t(last) ? x : uint32_t(last));
}

// Where the end of entry t is in an array of n starts with n ends behind them.
TT_HOST_DEVICE int64_t index_end(int32_t n, int32_t t) { return int64_t(n) + t; }

}  // namespace tt
