// sort_ids.hip -- ids by 32-bit keys, device-wide (gfx950).
#include <rocprim/iterator/counting_iterator.hpp>

#include "sort_config.hpp"

namespace tb {

static __global__ void k_ids_loaded() {}
void load_sort_ids(tribit_ctx* ctx) { load_code(ctx, kSortIdsFile, reinterpret_cast<const void*>(k_ids_loaded)); }

// order: the numbers of the items in the stable order of their keys' low `bits`
// bits. Keys of one 8-bit digit (octave classes) keep rocPRIM's own digits.
void sort_ids_device(tribit_ctx* ctx, const uint32_t* in, uint32_t* out, uint32_t* order, uint64_t n, uint32_t bits) {
  const auto sort = [&](auto config) {
    with_temp(ctx, [&](void* t, size_t& b) {
      return rocprim::radix_sort_pairs<decltype(config)>(t, b, in, out, rocprim::counting_iterator<uint32_t>(0), order,
                                                         (size_t)n, 0u, bits, ctx->stream);
    });
  };
  if (bits <= 8)
    with_sort_config<rocprim::default_config>(n, bits, sort);
  else
    with_sort_config<IdSortConfig>(n, bits, sort);
}

}  // namespace tb
