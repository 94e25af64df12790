// sort_records.hip -- 64-bit records by 32-bit keys, device-wide (gfx950).
#include "sort_config.hpp"

namespace tb {

static __global__ void k_records_loaded() {}
void load_sort_records(tribit_ctx* ctx) {
  load_code(ctx, kSortRecordsFile, reinterpret_cast<const void*>(k_records_loaded));
}

void sort_records_device(tribit_ctx* ctx, const uint32_t* in, uint32_t* out, const uint64_t* vin, uint64_t* vout,
                         uint64_t n, uint32_t bits) {
  with_sort_config<IdSortConfig>(n, bits, [&](auto config) {
    with_temp(ctx, [&](void* t, size_t& b) {
      return rocprim::radix_sort_pairs<decltype(config)>(t, b, in, out, vin, vout, (size_t)n, 0u, bits, ctx->stream);
    });
  });
}

}  // namespace tb
