// zero.hpp -- small device helpers of preprocessing: spans cleared by a kernel on
// the way, and scans by one workgroup.
#pragma once
#include <algorithm>

#include <rocprim/block/block_scan.hpp>

#include "common.hpp"

namespace tb {

// Ids in col16: m rounded up to whole dwords, and one more dword.
__host__ __device__ inline uint64_t col16_ids(uint64_t m) { return ((m + 1) / 2 + 1) * 2; }

// Zeroed on the way by a kernel over `items` of its own: one launch fewer each.
// A launch has fewer than 2^32 threads, so from 2^30 ids on a thread clears
// several words of the longest span (8 bytes an id).
struct ZeroSpans {
  uint32_t* p[3];
  uint64_t n[3];
  bool more = false;  // a span has more words than the launch has threads
  __device__ __forceinline__ void clear(uint64_t i) const {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (i < n[k]) p[k][i] = 0u;
    if (!more) return;
    const uint64_t threads = (uint64_t)gridDim.x * blockDim.x;
    for (int k = 0; k < 3; ++k)
      for (uint64_t j = i + threads; j < n[k]; j += threads) p[k][j] = 0u;
  }
  uint64_t grid_items(uint64_t items) {
    const uint64_t most = std::max(n[0], std::max(n[1], n[2]));
    const uint64_t all = std::max(items, std::min<uint64_t>(most, 1ull << 31));
    more = most > all;
    return all;
  }
};

// out[0, n]: the exclusive scan of f(0), ..., f(n - 1), by one workgroup in one
// launch (the device-wide scan takes two and is faster beyond kSmallScan items).
// Items change hands in LDS so that memory is read and written in whole lines:
// 5.4 us for 8192 items, 9.3 with eight neighbouring items per thread.
constexpr uint64_t kSmallScan = 32768;
constexpr uint32_t kScanBlockThreads = 1024;
constexpr uint32_t kScanBlockItems = 8;
template <typename F>
__device__ __forceinline__ void scan_block(const F& f, uint32_t n, uint32_t* __restrict__ out) {
  using Scan = rocprim::block_scan<uint32_t, kScanBlockThreads>;
  __shared__ typename Scan::storage_type tmp;
  __shared__ uint32_t buf[kScanBlockThreads * (kScanBlockItems + 1)];  // a dword of padding per thread
  uint32_t carry = 0;
  for (uint32_t i0 = 0; i0 < n; i0 += kScanBlockThreads * kScanBlockItems) {
    uint32_t v[kScanBlockItems], total;
#pragma unroll
    for (uint32_t j = 0; j < kScanBlockItems; ++j) {
      const uint32_t k = threadIdx.x + j * kScanBlockThreads;
      v[j] = i0 + k < n ? f(i0 + k) : 0u;
    }
#pragma unroll
    for (uint32_t j = 0; j < kScanBlockItems; ++j) {
      const uint32_t k = threadIdx.x + j * kScanBlockThreads;
      buf[k + k / kScanBlockItems] = v[j];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kScanBlockItems; ++j) v[j] = buf[threadIdx.x * (kScanBlockItems + 1) + j];
    Scan().exclusive_scan(v, v, carry, total, tmp, rocprim::plus<uint32_t>());
#pragma unroll
    for (uint32_t j = 0; j < kScanBlockItems; ++j) buf[threadIdx.x * (kScanBlockItems + 1) + j] = v[j];
    carry += total;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kScanBlockItems; ++j) {
      const uint32_t k = threadIdx.x + j * kScanBlockThreads;
      if (i0 + k < n) out[i0 + k] = buf[k + k / kScanBlockItems];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[n] = carry;
}

template <typename F>
__global__ void __launch_bounds__(kScanBlockThreads) k_scan_block(F f, uint32_t n, uint32_t* __restrict__ out) {
  scan_block(f, n, out);
}

}  // namespace tb
