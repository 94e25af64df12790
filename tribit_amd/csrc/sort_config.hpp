// sort_config.hpp -- rocPRIM's radix sorts of 32-bit ids with values: digits and tiles by size.
#pragma once
#include <rocprim/device/device_radix_sort.hpp>

#include "common.hpp"

namespace tb {

// 9-bit digits for the sorts of 32-bit ids (three passes instead of four for
// ids below 2^27). Measured on MI355X over 2^29 random 25-bit keys: pairs
// with 32-bit values 14.7 -> 11.5 ms, keys alone 9.6 -> 8.0 ms. The 64-bit
// key sorts keep rocPRIM's 8-bit digits (9 bits: 22.1 -> 23.4 ms; 10 bits
// slower still).
using IdSortConfig = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<1024, 16>, rocprim::kernel_config<1024, 16>, 9,
                                        rocprim::block_radix_rank_algorithm::match>>;
// rocPRIM merges blocks instead of sweeping digits up to 2^20 items: a launch per
// doubling, each over all items. Digits of 8 bits in small tiles (two or three
// passes of 7 to 14 us) are faster from kFewSort16 and kFewSort items on; whole builds with
// digits / with merges, us: 40K ids 65K edges 222 / 226, 100K 228 / 241, 300K 326 /
// 399, 1M 425 / 533; 1M ids 65K edges 291 / 344, 1M 546 / 703. Keys of more than 16
// bits take a third pass: 250K ids 40K edges 282 / 268, 160K 327 / 329. Beyond 2^20
// items the larger tiles of IdSortConfig win: 150K ids 4M edges 863 / 774.
constexpr uint64_t kFewSort16 = 1ull << 16, kFewSort = 1ull << 18, kFewSortEnd = 1ull << 20;
using FewSortConfig = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<512, 8>, rocprim::kernel_config<512, 8>, 8,
                                        rocprim::block_radix_rank_algorithm::match>,
    0>;

// sort(config) with the configuration for n items of `bits` bits: Large for many.
template <typename Large, typename F>
void with_sort_config(uint64_t n, uint32_t bits, F&& sort) {
  if (n <= kFewSortEnd && n >= (bits <= 16 ? kFewSort16 : kFewSort))
    sort(FewSortConfig{});
  else
    sort(Large{});
}

}  // namespace tb
