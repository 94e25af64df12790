// sort_keys.hip -- 64-bit keys sorted and made distinct, device-wide (gfx950).
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_select.hpp>

#include "common.hpp"

namespace tb {

static __global__ void k_keys_loaded() {}
void load_sort_keys(tribit_ctx* ctx) { load_code(ctx, kSortKeysFile, reinterpret_cast<const void*>(k_keys_loaded)); }

void sort_keys_device(tribit_ctx* ctx, const uint64_t* in, uint64_t* out, uint64_t n, uint32_t end_bit) {
  with_temp(ctx, [&](void* t, size_t& b) {
    return rocprim::radix_sort_keys(t, b, in, out, (size_t)n, 0u, end_bit, ctx->stream);
  });
}

// The sorted in[0, n) without repetitions into out, their number into *count (device memory).
void unique_device(tribit_ctx* ctx, const uint64_t* in, uint64_t* out, uint64_t* count, uint64_t n) {
  with_temp(ctx, [&](void* t, size_t& b) {
    return rocprim::unique(t, b, in, out, count, (size_t)n, rocprim::equal_to<uint64_t>(), ctx->stream);
  });
}

}  // namespace tb
