// ends.hpp -- how the endpoints of count_degrees are cut into counting tasks
// (host and device).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace tb {

// Endpoints per counting task: about two tasks per CU, between 2^17 (smaller
// ones spend their time adding 32K counters to memory: 1.1M edges over 200K ids
// 0.17 ms with 2^21) and 2^21.
inline uint32_t end_chunk(uint64_t m, uint32_t cus) {
  return (uint32_t)std::min<uint64_t>(1u << 21, std::max<uint64_t>(1u << 17, 2 * m / cus));
}

// Chunks of `chunk` endpoints that `ends` of one id group fill. Rounded up
// without a sum: a group may hold nearly 2^32 endpoints (a complete graph on its
// 65,536 ids: 4,294,901,760), to which adding the chunk wraps.
__host__ __device__ inline uint32_t end_chunks(uint32_t ends, uint32_t chunk) {
  return ends / chunk + (ends % chunk != 0 ? 1u : 0u);
}

}  // namespace tb
