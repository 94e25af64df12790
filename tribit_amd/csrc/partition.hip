// partition.hip -- preprocessing by partitioning instead of sorting (gfx950):
// distinct edge keys and vertex degrees.
//
// No counterpart in the reference, which sorts (src/single_gpu/tribit.cu:666).
// A radix sort of the 50-bit keys of R-MAT scale 25 streams them eight times
// through HBM; removing duplicates only needs equal keys to meet, so the keys
// are spread by a mixing bijection over buckets that fit in LDS, in one or two
// passes, and each bucket is made distinct in an LDS hash set. Degrees are
// counted the same way: endpoints spread by id range, counted in LDS. Measured
// at R-MAT scale 25 (537M keys): check, sort and removal of duplicates 28 ms ->
// 8.8 ms (3.2 + 1.8 + 3.7); degrees 13.9 (a sort of the larger endpoints, runs
// added by atomics) -> 4.5 ms.
#include <algorithm>

#include "common.hpp"
#include "device.hpp"
#include "ends.hpp"

namespace tb {

constexpr unsigned kBlock = 256;
constexpr uint32_t kPartThreads = 512;
constexpr uint32_t kPartItems = 12;                          // items per thread and tile
constexpr uint32_t kPartTile = kPartThreads * kPartItems;    // 48 KiB of 8-byte items: two blocks per CU

// A bijection of the W = 2 kb bit integers and its inverse (two rounds of xor
// shift and odd multiplier, as integer finalisers do; the multipliers are
// SplitMix64's, their inverses modulo 2^64 by Newton's iteration at compile
// time). Its high bits choose the bucket, so keys of any graph spread evenly.
constexpr uint64_t kMixA = 0xBF58476D1CE4E5B9ull, kMixB = 0x94D049BB133111EBull;
constexpr uint64_t mul_inverse(uint64_t a) {
  uint64_t x = a;  // correct to 3 bits; every step doubles that
  for (int i = 0; i < 5; ++i) x *= 2 - a * x;
  return x;
}
static_assert(kMixA * mul_inverse(kMixA) == 1 && kMixB * mul_inverse(kMixB) == 1, "inverses");

__host__ __device__ __forceinline__ uint64_t mix_key(uint64_t x, uint32_t kb, uint64_t mask) {
  x ^= x >> kb;
  x = (x * kMixA) & mask;
  x ^= x >> kb;
  x = (x * kMixB) & mask;
  return x ^ (x >> kb);
}
__host__ __device__ __forceinline__ uint64_t unmix_key(uint64_t x, uint32_t kb, uint64_t mask) {
  constexpr uint64_t ia = mul_inverse(kMixA), ib = mul_inverse(kMixB);
  x ^= x >> kb;  // the shift is at least half the width: its own inverse
  x = (x * ib) & mask;
  x ^= x >> kb;
  x = (x * ia) & mask;
  return x ^ (x >> kb);
}

// LDS state of one tile of a partition pass over nd digits.
struct SplitLds {
  uint32_t* hist;   // nd: items per digit, then the digit's first slot in the tile
  uint32_t* rel;    // nd: the digit's reserved place in its bucket minus its first slot
  uint32_t* wsum;   // one word per wave
};

// Exclusive scan of h[0, nd) in place by the whole block; returns the total.
__device__ __forceinline__ uint32_t block_scan(uint32_t* h, uint32_t nd, uint32_t* wsum) {
  const uint32_t per = (nd + kPartThreads - 1) / kPartThreads, i0 = threadIdx.x * per;
  uint32_t sum = 0;
  for (uint32_t i = i0; i < min(i0 + per, nd); ++i) sum += h[i];
  uint32_t inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o);
    if (lane_id() >= (uint32_t)o) inc += t;
  }
  if (lane_id() == 63) wsum[threadIdx.x >> 6] = inc;
  __syncthreads();
  uint32_t base = inc - sum, total = 0;
  for (uint32_t w = 0; w < kPartThreads / 64; ++w) {
    if (w < (threadIdx.x >> 6)) base += wsum[w];
    total += wsum[w];
  }
  for (uint32_t i = i0; i < min(i0 + per, nd); ++i) {
    const uint32_t c = h[i];
    h[i] = base;
    base += c;
  }
  __syncthreads();
  return total;
}

// Whether a bucket overflowed (bit 1 of *flags): what is left of the partition is
// then work for nothing. Best effort, one relaxed read per block (by every wave of
// k_distinct, whose total is in the same line, it took 0.17 ms).
__device__ __forceinline__ bool overflowed(const uint32_t* flags) {
  return (__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 2u) != 0;
}

// Keys (min << 32) | max: checked (min < max < n, else *flags |= 1), sentinels
// dropped, packed to W = 2 kb bits, mixed and spread by the high `bits` bits
// over buckets of `cap` items (cursor: items per bucket; *flags |= 2 when one
// overflows, whose items past the end are dropped, and later tiles with them).
//
// Bound by memory (16 bytes a key). A tile is grouped by digit in LDS first, so
// a bucket receives runs of tile / 2^bits items (96 bytes at 512 buckets) from
// one reservation instead of single keys.
__global__ void __launch_bounds__(kPartThreads) k_split_keys(const uint64_t* __restrict__ keys, uint64_t nk,
                                                             uint64_t n, uint32_t kb, uint32_t bits, uint64_t cap,
                                                             uint64_t* __restrict__ out, uint32_t* __restrict__ cursor,
                                                             uint32_t* __restrict__ flags) {
  __shared__ uint64_t s_item[kPartTile];
  __shared__ uint16_t s_dig[kPartTile];
  __shared__ uint32_t s_wsum[kPartThreads / 64];
  __shared__ bool s_stop;
  extern __shared__ uint32_t s_dyn[];
  const uint32_t nd = 1u << bits;
  uint32_t *hist = s_dyn, *rel = s_dyn + nd;
  if (threadIdx.x == 0) s_stop = overflowed(flags);
  const uint32_t W = 2 * kb;
  const uint64_t mask = W >= 64 ? ~0ull : (1ull << W) - 1;
  const uint32_t shift = W - bits;
  for (uint32_t i = threadIdx.x; i < nd; i += kPartThreads) hist[i] = 0u;
  __syncthreads();
  if (s_stop) return;
  uint64_t h[kPartItems];
  uint32_t dr[kPartItems];  // digit << 16 | rank in the tile; all ones: no item
  bool bad = false;
  const uint64_t i0 = (uint64_t)blockIdx.x * kPartTile + threadIdx.x;
#pragma unroll
  for (uint32_t j = 0; j < kPartItems; ++j) {
    const uint64_t i = i0 + (uint64_t)j * kPartThreads;
    h[j] = i < nk ? keys[i] : kSentinel;
  }
#pragma unroll
  for (uint32_t j = 0; j < kPartItems; ++j) {
    const uint64_t a = h[j] >> 32, b = h[j] & 0xFFFFFFFFull;
    const bool have = h[j] != kSentinel, ok = a < b && b < n;
    bad |= have && !ok;
    dr[j] = 0xFFFFFFFFu;
    if (have && ok) {
      h[j] = mix_key((a << kb) | b, kb, mask);
      const uint32_t d = shift < 64 ? (uint32_t)(h[j] >> shift) : 0u;
      dr[j] = (d << 16) | atomicAdd(&hist[d], 1u);
    }
  }
  if (__any(bad) && lane_id() == 0) atomicOr(flags, 1u);
  __syncthreads();
  // reserve each digit's run in its bucket, then its slots in the tile
  for (uint32_t d = threadIdx.x; d < nd; d += kPartThreads) {
    const uint32_t c = hist[d];
    uint32_t at = 0;
    if (c) {
      at = atomicAdd(&cursor[d], c);
      if ((uint64_t)at + c > cap) atomicOr(flags, 2u);
    }
    rel[d] = at;
  }
  __syncthreads();
  const uint32_t total = block_scan(hist, nd, s_wsum);
  for (uint32_t d = threadIdx.x; d < nd; d += kPartThreads) rel[d] -= hist[d];
#pragma unroll
  for (uint32_t j = 0; j < kPartItems; ++j)
    if (dr[j] != 0xFFFFFFFFu) {
      const uint32_t at = hist[dr[j] >> 16] + (dr[j] & 0xFFFFu);
      s_item[at] = h[j];
      s_dig[at] = (uint16_t)(dr[j] >> 16);
    }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kPartThreads) {
    const uint32_t d = s_dig[i], at = rel[d] + i;
    if (at < cap) out[(uint64_t)d * cap + at] = s_item[i];
  }
}

// The second pass: bucket blockIdx.y of the first, tile blockIdx.x, spread by
// the next `bits` bits below `shift` + bits; of the mixed key only its low
// `shift` bits are kept (P = uint32_t when they fit: half the bytes from here).
template <typename P>
__global__ void __launch_bounds__(kPartThreads) k_split_bucket(const uint64_t* __restrict__ in, uint64_t cap1,
                                                               const uint32_t* __restrict__ cnt1, uint32_t bits,
                                                               uint32_t shift, uint32_t cap, P* __restrict__ out,
                                                               uint32_t* __restrict__ cursor,
                                                               uint32_t* __restrict__ flags) {
  __shared__ P s_item[kPartTile];
  __shared__ uint16_t s_dig[kPartTile];
  __shared__ uint32_t s_wsum[kPartThreads / 64];
  __shared__ bool s_stop;
  extern __shared__ uint32_t s_dyn[];
  const uint32_t nd = 1u << bits, b1 = blockIdx.y;
  const uint64_t cnt = min((uint64_t)cnt1[b1], cap1);
  const uint64_t t0 = (uint64_t)blockIdx.x * kPartTile;
  if (t0 >= cnt) return;
  uint32_t *hist = s_dyn, *rel = s_dyn + nd;
  if (threadIdx.x == 0) s_stop = overflowed(flags);
  for (uint32_t i = threadIdx.x; i < nd; i += kPartThreads) hist[i] = 0u;
  __syncthreads();
  if (s_stop) return;
  in += (uint64_t)b1 * cap1;
  cursor += (uint64_t)b1 * nd;
  out += (uint64_t)b1 * nd * cap;
  const uint64_t low = (1ull << shift) - 1;  // shift <= 63 - bits
  uint64_t h[kPartItems];
  uint32_t dr[kPartItems];
#pragma unroll
  for (uint32_t j = 0; j < kPartItems; ++j) {
    const uint64_t i = t0 + threadIdx.x + j * kPartThreads;
    h[j] = i < cnt ? in[i] : 0ull;
    dr[j] = i < cnt ? 0u : 0xFFFFFFFFu;
  }
#pragma unroll
  for (uint32_t j = 0; j < kPartItems; ++j)
    if (dr[j] == 0u) {
      const uint32_t d = (uint32_t)(h[j] >> shift) & (nd - 1);
      dr[j] = (d << 16) | atomicAdd(&hist[d], 1u);
    }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < nd; d += kPartThreads) {
    const uint32_t c = hist[d];
    uint32_t at = 0;
    if (c) {
      at = atomicAdd(&cursor[d], c);
      if (at + c > cap) atomicOr(flags, 2u);
    }
    rel[d] = at;
  }
  __syncthreads();
  const uint32_t total = block_scan(hist, nd, s_wsum);
  for (uint32_t d = threadIdx.x; d < nd; d += kPartThreads) rel[d] -= hist[d];
#pragma unroll
  for (uint32_t j = 0; j < kPartItems; ++j)
    if (dr[j] != 0xFFFFFFFFu) {
      const uint32_t at = hist[dr[j] >> 16] + (dr[j] & 0xFFFFu);
      s_item[at] = (P)(h[j] & low);
      s_dig[at] = (uint16_t)(dr[j] >> 16);
    }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kPartThreads) {
    const uint32_t d = s_dig[i], at = rel[d] + i;
    if (at < cap) out[(uint64_t)d * cap + at] = s_item[i];
  }
}

// Final buckets: at most kBucketCap items each (1,024 to 2,048 on average, so
// that only inputs with heavily repeated keys overflow one).
constexpr uint32_t kBucketCap = 3072;
constexpr uint32_t kBucketAvg = 2048;
constexpr uint32_t kSetSlots = 4096;

__device__ __forceinline__ uint32_t cas_slot(uint32_t* p, uint32_t x) { return atomicCAS(p, 0xFFFFFFFFu, x); }
__device__ __forceinline__ uint64_t cas_slot(uint64_t* p, uint64_t x) {
  return atomicCAS(reinterpret_cast<unsigned long long*>(p), ~0ull, (unsigned long long)x);
}

// Distinct keys of `nb` buckets: an LDS hash set per bucket (open addressing,
// at most 3/4 full), its new members appended to an LDS list, the lists of GROUP
// buckets written out together with one reservation in `out` (one atomic on the
// shared total per bucket would serialise at about 13 ns each). The all-ones
// item marks a free slot, so its own presence is a flag. Also counts the keys
// that join ids less than `band_ids` apart into *band (when given).
template <typename P, uint32_t GROUP>
__global__ void __launch_bounds__(kPartThreads) k_distinct(const P* __restrict__ in, uint64_t cap,
                                                           const uint32_t* __restrict__ cnt, uint32_t nb, uint32_t kb,
                                                           uint32_t rbits, uint64_t* __restrict__ out,
                                                           const uint32_t* __restrict__ flags,
                                                           uint32_t* __restrict__ total, uint64_t band_ids,
                                                           unsigned long long* __restrict__ band) {
  if (*flags & 2u) return;  // set before this launch or not at all: a plain read, beside the total's atomics
  constexpr P kFree = (P)~(P)0;
  __shared__ P s_set[kSetSlots];
  __shared__ P s_list[GROUP * kBucketCap];
  __shared__ uint32_t s_n, s_ones, s_base, s_off[GROUP + 1];
  const uint32_t W = 2 * kb, lane = lane_id();
  const uint64_t mask = W >= 64 ? ~0ull : (1ull << W) - 1, lo = (1ull << kb) - 1;
  uint64_t acc = 0;
  for (uint32_t g = blockIdx.x; (uint64_t)g * GROUP < nb; g += gridDim.x) {
    const uint32_t b0 = g * GROUP, nq = min(GROUP, nb - b0);
    if (threadIdx.x == 0) s_n = 0;
    for (uint32_t q = 0; q < nq; ++q) {
      const uint32_t c = min((uint64_t)cnt[b0 + q], min(cap, (uint64_t)kBucketCap));
      const P* src = in + (uint64_t)(b0 + q) * cap;
      for (uint32_t i = threadIdx.x; i < kSetSlots; i += kPartThreads) s_set[i] = kFree;
      if (threadIdx.x == 0) {
        s_ones = 0;
        s_off[q] = s_n;  // every append of the bucket before is behind a barrier
      }
      __syncthreads();
      for (uint32_t i0 = 0; i0 < c; i0 += kPartThreads) {  // block-uniform
        const uint32_t i = i0 + threadIdx.x;
        bool fresh = false;
        P x = 0;
        if (i < c) {
          x = src[i];
          if (x == kFree) {
            fresh = atomicExch(&s_ones, 1u) == 0u;
          } else {
            uint32_t at = ((uint32_t)x ^ (uint32_t)((uint64_t)x >> 20)) & (kSetSlots - 1);
            for (;;) {  // fewer members than slots: ends at the key or a free slot
              const P y = cas_slot(&s_set[at], x);
              fresh = y == kFree;
              if (fresh || y == x) break;
              at = (at + 1) & (kSetSlots - 1);
            }
          }
        }
        const uint64_t m = __ballot(fresh);
        uint32_t base = 0;
        if (lane == 0 && m) base = atomicAdd(&s_n, (uint32_t)__popcll(m));
        base = __shfl(base, 0);
        if (fresh) s_list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = x;
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      s_off[nq] = s_n;
      s_base = s_n ? atomicAdd(total, s_n) : 0u;
    }
    __syncthreads();
    for (uint32_t q = 0; q < nq; ++q) {
      const uint64_t high = rbits < 64 ? (uint64_t)(b0 + q) << rbits : 0ull;
      for (uint32_t i = s_off[q] + threadIdx.x; i < s_off[q + 1]; i += kPartThreads) {
        const uint64_t k = unmix_key(high | (uint64_t)s_list[i], kb, mask);
        out[s_base + i] = k;
        acc += (k & lo) - (k >> kb) < band_ids;
      }
    }
    __syncthreads();
  }
  if (!band) return;
  acc = wave_sum_u64(acc);
  if (lane == 0 && acc) atomicAdd(band, (unsigned long long)acc);
}

__global__ void k_part_zero(uint32_t* __restrict__ p, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// Distinct keys of d_keys (as given, (min << 32) | max with sentinels), packed
// (min << kb) | max, in any order, into out (room for nk). One device read-back.
// Returns false when a bucket overflowed (keys repeated so often that hashing
// cannot spread them): nothing is in `out` then, and the caller sorts. The passes
// end early then: the 300M keys of 100K edges cost the time of the first one.
bool distinct_keys(tribit_ctx* ctx, const uint64_t* d_keys, uint64_t nk, uint64_t n, uint32_t kb, uint64_t* out,
                   uint64_t* m, bool* bad, uint64_t band_ids, uint64_t* band) {
  hipStream_t s = ctx->stream;
  const uint32_t W = 2 * kb;
  uint32_t B = 0;  // bits of the final bucket number
  while (((nk + kBucketAvg - 1) / kBucketAvg) > (1ull << B)) ++B;
  B = std::min(B, W);
  const bool two = B > 9;
  const uint32_t b1 = two ? (B + 1) / 2 : B, b2 = B - b1, r = W - B;
  const uint32_t nd1 = 1u << b1;
  const uint64_t nb = 1ull << B;
  const uint64_t cap1 = two ? nk / nd1 + nk / nd1 / 8 + 4096 : kBucketCap;
  DevBuf<uint64_t> reg1(ctx, cap1 * nd1);
  // cursors of both passes, then: flags, total, band (two words)
  const uint64_t words = ((nd1 + (two ? nb : 0) + 1) & ~1ull) + 4;
  DevBuf<uint32_t> cur(ctx, words);
  uint32_t* tail = cur.p + (words - 4);  // 8-byte aligned
  k_part_zero<<<grid_for(words, kBlock), kBlock, 0, s>>>(cur.p, words);
  k_split_keys<<<grid_for(nk, kPartTile), kPartThreads, 8 * nd1, s>>>(d_keys, nk, n, kb, b1, cap1, reg1.p, cur.p,
                                                                     tail);
  unsigned long long* d_band = reinterpret_cast<unsigned long long*>(tail + 2);
  const uint32_t cus = (uint32_t)(ctx->cus > 0 ? ctx->cus : 256);
  DevBuf<uint32_t> reg4;
  DevBuf<uint64_t> reg8;
  if (two) {
    const dim3 grid(grid_for(cap1, kPartTile), nd1);
    const uint32_t nd2 = 1u << b2;
    if (r <= 32) {
      reg4 = DevBuf<uint32_t>(ctx, nb * kBucketCap);
      k_split_bucket<uint32_t><<<grid, kPartThreads, 8 * nd2, s>>>(reg1.p, cap1, cur.p, b2, r, kBucketCap, reg4.p,
                                                                 cur.p + nd1, tail);
      reg1.reset();
      k_distinct<uint32_t, 4><<<std::min<uint32_t>(grid_for(nb, 4), 8 * cus), kPartThreads, 0, s>>>(
          reg4.p, kBucketCap, cur.p + nd1, (uint32_t)nb, kb, r, out, tail, tail + 1, band_ids, band ? d_band : nullptr);
    } else {
      reg8 = DevBuf<uint64_t>(ctx, nb * kBucketCap);
      k_split_bucket<uint64_t><<<grid, kPartThreads, 8 * nd2, s>>>(reg1.p, cap1, cur.p, b2, r, kBucketCap, reg8.p,
                                                                 cur.p + nd1, tail);
      reg1.reset();
      k_distinct<uint64_t, 1><<<std::min<uint32_t>((uint32_t)nb, 8 * cus), kPartThreads, 0, s>>>(
          reg8.p, kBucketCap, cur.p + nd1, (uint32_t)nb, kb, r, out, tail, tail + 1, band_ids, band ? d_band : nullptr);
    }
  } else {
    // the first pass kept whole mixed keys: the bucket bits are already in them
    k_distinct<uint64_t, 1><<<std::min<uint32_t>((uint32_t)nb, 8 * cus), kPartThreads, 0, s>>>(
        reg1.p, cap1, cur.p, (uint32_t)nb, kb, 64, out, tail, tail + 1, band_ids, band ? d_band : nullptr);
  }
  uint32_t h[4] = {0, 0, 0, 0};
  TB_HIP(hipMemcpyAsync(h, tail, sizeof(h), hipMemcpyDeviceToHost, s));
  ctx->sync();
  TB_HIP(hipGetLastError());
  *bad = h[0] & 1u;
  *m = h[1];
  if (band) *band = (uint64_t)h[2] | ((uint64_t)h[3] << 32);
  return !(h[0] & 2u) || *bad;
}

// ---------------------------------------------------------------- degrees
// deg[v] = how often v is an endpoint of the keys (lo << kb) | hi. One atomic
// per endpoint reaches 14 G/s (37 ms for the 523M keys of R-MAT scale 25), so
// beyond kDirectEdges keys the endpoints' low 16 bits are first grouped by
// their high bits (2 bytes written per endpoint), and each group of 65,536 ids
// is counted in LDS, half of its ids at a time. A pass covers up to
// kEndMaxGroups groups (2^27 ids), so that a tile's runs stay long, and up to
// kEndSpan keys, so that 32 bits hold a group's endpoints.
constexpr uint64_t kDirectEdges = 1ull << 18;
constexpr uint32_t kEndBits = 16;
constexpr uint32_t kEndMaxGroups = 2048;
constexpr uint64_t kEndSpan = 0x7FFFFFFF;
constexpr uint32_t kEndKeys = 16;         // keys per thread and tile: 32 KiB of halves, as much of digits
constexpr uint32_t kEndTile = kPartThreads * kEndKeys;
constexpr uint32_t kEndCounters = 32768;  // 128 KiB of LDS
constexpr uint32_t kEndThreads = 1024;

// Few edges over more ids than LDS holds: a block counts the first id that comes
// to each slot of a direct-mapped table in LDS, and adds the others one by one. A
// hub comes often, so some other id keeps it out of its slot in few blocks. With
// an atomic per endpoint a star of 2^18 edges queued on one address (its build
// 3.3 ms; a random graph's of that size 0.33).
constexpr uint32_t kTableSlots = 4096;
constexpr uint32_t kTableKeys = 2;  // keys per thread
__global__ void __launch_bounds__(kEndThreads) k_deg_table(const uint64_t* __restrict__ keys, uint32_t m, uint32_t kb,
                                                           uint32_t* __restrict__ deg) {
  constexpr uint32_t kFree = 0xFFFFFFFFu;  // ids are below 2^32 - 2
  __shared__ uint32_t s_id[kTableSlots], s_n[kTableSlots];
  for (uint32_t i = threadIdx.x; i < kTableSlots; i += kEndThreads) {
    s_id[i] = kFree;
    s_n[i] = 0u;
  }
  __syncthreads();
  const uint64_t lo = (1ull << kb) - 1;
  const auto add = [&](uint32_t v) {
    const uint32_t at = (v * 0x9E3779B1u) >> 20;
    const uint32_t owner = atomicCAS(&s_id[at], kFree, v);
    if (owner == kFree || owner == v)
      atomicAdd(&s_n[at], 1u);
    else
      atomicAdd(&deg[v], 1u);
  };
#pragma unroll
  for (uint32_t j = 0; j < kTableKeys; ++j) {
    const uint32_t i = (blockIdx.x * kTableKeys + j) * kEndThreads + threadIdx.x;
    if (i < m) {
      const uint64_t k = keys[i];
      add((uint32_t)(k >> kb));
      add((uint32_t)(k & lo));
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kTableSlots; i += kEndThreads)
    if (s_n[i]) atomicAdd(&deg[s_id[i]], s_n[i]);
}

// Few edges over ids that fit LDS: every block counts its share there and adds
// it once (80K edges of an R-MAT graph, whose hubs' atomics queue up: 45 us with
// an atomic per endpoint).
__global__ void __launch_bounds__(kEndThreads) k_deg_lds(const uint64_t* __restrict__ keys, uint32_t m, uint32_t kb,
                                                         uint32_t n, uint32_t* __restrict__ deg) {
  __shared__ uint32_t s_c[kEndCounters];
  for (uint32_t i = threadIdx.x; i < n; i += kEndThreads) s_c[i] = 0u;
  __syncthreads();
  const uint64_t lo = (1ull << kb) - 1;
  for (uint32_t i = blockIdx.x * kEndThreads + threadIdx.x; i < m; i += gridDim.x * kEndThreads) {
    const uint64_t k = keys[i];
    atomicAdd(&s_c[(uint32_t)(k >> kb)], 1u);
    atomicAdd(&s_c[(uint32_t)(k & lo)], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += kEndThreads)
    if (s_c[i]) atomicAdd(&deg[i], s_c[i]);
}

__global__ void __launch_bounds__(kPartThreads) k_ends_hist(const uint64_t* __restrict__ keys, uint64_t m, uint32_t kb,
                                                            uint32_t g0, uint32_t groups,
                                                            uint32_t* __restrict__ hist) {
  extern __shared__ uint32_t s_h[];
  for (uint32_t i = threadIdx.x; i < groups; i += blockDim.x) s_h[i] = 0u;
  __syncthreads();
  const uint64_t lo = (1ull << kb) - 1;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t k = keys[i];
    const uint32_t ga = ((uint32_t)(k >> kb) >> kEndBits) - g0, gb = ((uint32_t)(k & lo) >> kEndBits) - g0;
    if (ga < groups) atomicAdd(&s_h[ga], 1u);
    if (gb < groups) atomicAdd(&s_h[gb], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < groups; i += blockDim.x)
    if (s_h[i]) atomicAdd(&hist[i], s_h[i]);
}

// base[g]: the group's first endpoint (64 bits: 2 m may pass 2^32); task[g]: its
// first counting task (two per chunk of `chunk` endpoints). One block.
__global__ void __launch_bounds__(kPartThreads) k_ends_base(const uint32_t* __restrict__ hist, uint32_t groups,
                                                            uint32_t chunk,
                                                            uint64_t* __restrict__ base, uint32_t* __restrict__ task) {
  __shared__ uint64_t s_b[kPartThreads];
  __shared__ uint32_t s_t[kPartThreads];
  const uint32_t per = (groups + kPartThreads - 1) / kPartThreads, i0 = threadIdx.x * per;
  uint64_t b = 0;
  uint32_t t = 0;
  for (uint32_t i = i0; i < min(i0 + per, groups); ++i) {
    b += hist[i];
    t += 2 * end_chunks(hist[i], chunk);
  }
  s_b[threadIdx.x] = b;
  s_t[threadIdx.x] = t;
  __syncthreads();
  uint64_t pb = 0;
  uint32_t pt = 0;
  for (uint32_t i = 0; i < threadIdx.x; ++i) {
    pb += s_b[i];
    pt += s_t[i];
  }
  for (uint32_t i = i0; i < min(i0 + per, groups); ++i) {
    base[i] = pb;
    task[i] = pt;
    pb += hist[i];
    pt += 2 * end_chunks(hist[i], chunk);
  }
  if (i0 < groups && i0 + per >= groups) {
    base[groups] = pb;
    task[groups] = pt;
  }
}

__global__ void __launch_bounds__(kPartThreads) k_ends_split(const uint64_t* __restrict__ keys, uint64_t m,
                                                             uint32_t kb, uint32_t g0, uint32_t groups,
                                                             const uint64_t* __restrict__ base,
                                                             uint32_t* __restrict__ cursor,
                                                             uint16_t* __restrict__ out) {
  __shared__ uint32_t s_item[2 * kEndTile];  // (group - g0) << 16 | low half
  __shared__ uint32_t s_wsum[kPartThreads / 64];
  extern __shared__ uint32_t s_dyn[];
  uint32_t *hist = s_dyn, *rel = s_dyn + groups;
  for (uint32_t i = threadIdx.x; i < groups; i += kPartThreads) hist[i] = 0u;
  __syncthreads();
  const uint64_t lo = (1ull << kb) - 1, i0 = (uint64_t)blockIdx.x * kEndTile + threadIdx.x;
  uint32_t a[kEndKeys], b[kEndKeys], ranks[kEndKeys];  // ranks: of a, and of b << 16 (a tile has 2^14 endpoints)
#pragma unroll
  for (uint32_t j = 0; j < kEndKeys; ++j) {
    const uint64_t i = i0 + (uint64_t)j * kPartThreads;
    const uint64_t k = i < m ? keys[i] : 0ull;
    // ids relative to the window; past it (or no key): all ones, whose group is no group
    a[j] = (uint32_t)(k >> kb) - (g0 << kEndBits);
    b[j] = (uint32_t)(k & lo) - (g0 << kEndBits);
    if (i >= m || a[j] >> kEndBits >= groups) a[j] = 0xFFFFFFFFu;
    if (i >= m || b[j] >> kEndBits >= groups) b[j] = 0xFFFFFFFFu;
  }
#pragma unroll
  for (uint32_t j = 0; j < kEndKeys; ++j) {
    ranks[j] = 0;
    if (a[j] != 0xFFFFFFFFu) ranks[j] = atomicAdd(&hist[a[j] >> kEndBits], 1u);
    if (b[j] != 0xFFFFFFFFu) ranks[j] |= atomicAdd(&hist[b[j] >> kEndBits], 1u) << 16;
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < groups; d += kPartThreads) rel[d] = hist[d] ? atomicAdd(&cursor[d], hist[d]) : 0u;
  __syncthreads();
  const uint32_t total = block_scan(hist, groups, s_wsum);
  for (uint32_t d = threadIdx.x; d < groups; d += kPartThreads) rel[d] -= hist[d];
#pragma unroll
  for (uint32_t j = 0; j < kEndKeys; ++j) {
    if (a[j] != 0xFFFFFFFFu) s_item[hist[a[j] >> kEndBits] + (ranks[j] & 0xFFFFu)] = a[j];
    if (b[j] != 0xFFFFFFFFu) s_item[hist[b[j] >> kEndBits] + (ranks[j] >> 16)] = b[j];
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kPartThreads) {
    const uint32_t x = s_item[i], d = x >> kEndBits;
    out[base[d] + (uint32_t)(rel[d] + i)] = (uint16_t)x;
  }
}

// Counting tasks: chunk c of group g, half h of its ids. A group of one chunk
// stores its counts, unless `more` spans of keys add to them; several chunks add
// theirs (deg is zero before).
__global__ void __launch_bounds__(kEndThreads) k_ends_count(const uint16_t* __restrict__ ends,
                                                            const uint64_t* __restrict__ base,
                                                            const uint32_t* __restrict__ task, uint32_t g0,
                                                            uint32_t groups, uint32_t chunk, uint64_t n, bool more,
                                                            uint32_t* __restrict__ deg) {
  __shared__ uint32_t s_c[kEndCounters];
  const uint32_t tasks = task[groups];
  for (uint32_t t = blockIdx.x; t < tasks; t += gridDim.x) {
    uint32_t lo = 0, hi = groups;  // task[lo] <= t < task[hi]
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (task[mid] <= t)
        lo = mid;
      else
        hi = mid;
    }
    const uint32_t g = lo, half = (t - task[g]) & 1u, c = (t - task[g]) >> 1;
    const bool sole = !more && task[g + 1] - task[g] == 2;
    for (uint32_t i = threadIdx.x; i < kEndCounters; i += kEndThreads) s_c[i] = 0u;
    __syncthreads();
    const uint64_t e0 = base[g] + (uint64_t)c * chunk, e1 = min(base[g + 1], e0 + chunk);
    // eight halves per 16-byte load; ends is padded past its last endpoint
    const uint64_t v0 = e0 / 8, v1 = (e1 + 7) / 8;
    const uint4* in = reinterpret_cast<const uint4*>(ends);
    for (uint64_t v = v0 + threadIdx.x; v < v1; v += kEndThreads) {
      const uint4 w = in[v];
      const uint32_t word[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (uint32_t k = 0; k < 8; ++k) {
        const uint32_t x = (word[k / 2] >> (16 * (k & 1))) & 0xFFFFu;
        const uint64_t e = 8 * v + k;
        if (e >= e0 && e < e1 && (x >> 15) == half) atomicAdd(&s_c[x & 0x7FFFu], 1u);
      }
    }
    __syncthreads();
    const uint64_t id0 = ((uint64_t)(g0 + g) << kEndBits) + (uint64_t)half * kEndCounters;
    for (uint32_t i = threadIdx.x; i < kEndCounters; i += kEndThreads) {
      const uint64_t id = id0 + i;
      if (id < n && s_c[i]) {
        if (sole)
          deg[id] = s_c[i];
        else
          atomicAdd(&deg[id], s_c[i]);
      }
    }
    __syncthreads();
  }
}

void count_degrees(tribit_ctx* ctx, const uint64_t* keys, uint64_t m, uint64_t n, uint32_t kb, uint32_t* deg) {
  hipStream_t s = ctx->stream;
  k_part_zero<<<grid_for(n, kBlock), kBlock, 0, s>>>(deg, n);
  if (!m) return;
  if (m <= kDirectEdges && n <= kEndCounters) {
    k_deg_lds<<<std::min<uint32_t>(64, grid_for(m, 4 * kEndThreads)), kEndThreads, 0, s>>>(keys, (uint32_t)m, kb,
                                                                                          (uint32_t)n, deg);
    return;
  }
  if (m <= kDirectEdges) {
    k_deg_table<<<grid_for(m, kTableKeys * kEndThreads), kEndThreads, 0, s>>>(keys, (uint32_t)m, kb, deg);
    return;
  }
  const uint32_t groups = (uint32_t)((n + (1ull << kEndBits) - 1) >> kEndBits);
  const uint32_t most = std::min(groups, kEndMaxGroups), cus = (uint32_t)(ctx->cus > 0 ? ctx->cus : 256);
  DevBuf<uint16_t> ends(ctx, 2 * std::min(m, kEndSpan) + 8);
  DevBuf<uint32_t> hist(ctx, 3 * most + 1);  // histogram, cursors, tasks
  DevBuf<uint64_t> base(ctx, most + 1);
  uint32_t *cursor = hist.p + most, *task = hist.p + 2 * most;
  for (uint64_t k0 = 0; k0 < m; k0 += kEndSpan) {
    const uint64_t* k = keys + k0;
    const uint64_t mk = std::min(m - k0, kEndSpan);
    const uint32_t chunk = end_chunk(mk, cus);
    for (uint32_t g0 = 0; g0 < groups; g0 += kEndMaxGroups) {
      const uint32_t ng = std::min(groups - g0, kEndMaxGroups);
      k_part_zero<<<grid_for(2 * most, kBlock), kBlock, 0, s>>>(hist.p, 2 * most);
      k_ends_hist<<<std::min<uint32_t>(4 * cus, grid_for(mk, kPartThreads)), kPartThreads, 4 * ng, s>>>(k, mk, kb, g0,
                                                                                                       ng, hist.p);
      k_ends_base<<<1, kPartThreads, 0, s>>>(hist.p, ng, chunk, base.p, task);
      k_ends_split<<<grid_for(mk, kEndTile), kPartThreads, 8 * ng, s>>>(k, mk, kb, g0, ng, base.p, cursor, ends.p);
      k_ends_count<<<cus, kEndThreads, 0, s>>>(ends.p, base.p, task, g0, ng, chunk, n, m > kEndSpan, deg);
    }
  }
}

}  // namespace tb
