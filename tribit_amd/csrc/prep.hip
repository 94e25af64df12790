// prep.hip -- on-GPU generators and preprocessing (edge keys in HBM ->
// degree-oriented int32 CSR, per-row wedge counts, streamed-range lists), gfx950.
//
// Replaces the reference's preprocessing chain, src/single_gpu/tribit.cu:
// 664-763 (radix sort + unique of packed keys, L/U bit structures, singleton
// purge, warp schedule). The product here is a degree-oriented CSR instead:
//   keys (min<<32|max) --partition, LDS hash sets--> m undirected edges
//   deg[v] (endpoints by id range, counted in LDS)
//   orient {a<b}: a->b iff deg(a) <= deg(b)       (rank = (deg, id))
//   --rows by partition, else a sort--> row_ptr[n+1] (u32), col[m] (u32, ascending
//   within a row)
//   W+ = sum over v of indeg(v) * outdeg(v); wedge ranges (relabelled graphs)
// Launches are 1-D grids of 256-thread blocks (4 waves); sorts and scans by one
// workgroup take 1024 threads.
#include <cmath>
#include <cstring>
#include <rocprim/block/block_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include "common.hpp"
#include "device.hpp"
#include "zero.hpp"

namespace tb {

constexpr unsigned kBlock = 256;

// ---------------------------------------------------------------- generators

// Bound by integer arithmetic (13 mix64 words and 25 quadrant draws per key at
// scale 25), not by its 8 bytes of output. The word index e * 16 + j advances by
// one per word, so the counter is one 64-bit add per word; both endpoints are 32
// bits (scale <= 31) and grow by an add with carry per level: src takes the
// predicate r >= t1, and dst the parity of r >= t0, r >= t1, r >= t2, which for
// t0 <= t1 <= t2 is 1 exactly in quadrants (0,1) and (1,1). 537M keys of scale
// 25: 9.75 -> 6.25 ms against a multiply per word and 64-bit endpoints.
__global__ void k_gen_rmat(uint64_t* __restrict__ keys, uint64_t ne, uint32_t scale, uint32_t t0, uint32_t t1,
                           uint32_t t2, uint64_t key) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < ne; e += stride) {
    uint32_t src = 0, dst = 0;
    uint64_t c = key + (e * 16) * kRandStep;  // rand_word(key, e * 16 + j) = mix64(c + j * kRandStep)
    auto level = [&](uint32_t r) {
      const bool g0 = r >= t0, g1 = r >= t1, g2 = r >= t2;
      src += src + (g1 ? 1u : 0u);
      dst += dst + ((g0 != (g1 != g2)) ? 1u : 0u);
    };
    for (uint32_t l = 0; l + 1 < scale; l += 2, c += kRandStep) {
      const uint64_t w = mix64(c);
      level((uint32_t)w);
      level((uint32_t)(w >> 32));
    }
    if (scale & 1) level((uint32_t)mix64(c));
    keys[e] = (src == dst) ? kSentinel
                           : (src < dst ? (((uint64_t)src << 32) | dst) : (((uint64_t)dst << 32) | src));
  }
}

__global__ void k_gen_er(uint64_t* __restrict__ keys, uint64_t ne, uint64_t n, uint64_t key) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < ne; e += stride) {
    const uint64_t w = rand_word(key, e);
    const uint64_t u = ((w & 0xFFFFFFFFull) * n) >> 32;
    const uint64_t v = ((w >> 32) * n) >> 32;
    keys[e] = (u == v) ? kSentinel : (u < v ? ((u << 32) | v) : ((v << 32) | u));
  }
}

void rmat_thresholds(double a, double b, double c, uint32_t t[3]) {
  const double two32 = 4294967296.0;
  const double s[3] = {a, a + b, a + b + c};
  for (int i = 0; i < 3; ++i) {
    double v = s[i] * two32;
    if (v < 0) v = 0;
    if (v > 4294967295.0) v = 4294967295.0;
    t[i] = (uint32_t)v;
  }
}

static unsigned gen_grid(tribit_ctx* ctx, uint64_t ne) {
  uint64_t g = (ne + kBlock - 1) / kBlock;
  const uint64_t cap = (uint64_t)(ctx->cus > 0 ? ctx->cus : 256) * 64;
  return (unsigned)(g < 1 ? 1 : (g > cap ? cap : g));
}

void gen_rmat(tribit_ctx* ctx, uint32_t scale, uint32_t ef, double a, double b, double c, uint64_t seed,
              uint64_t* d_keys) {
  uint32_t t[3];
  rmat_thresholds(a, b, c, t);
  const uint64_t ne = (uint64_t)ef << scale;
  k_gen_rmat<<<gen_grid(ctx, ne), kBlock, 0, ctx->stream>>>(d_keys, ne, scale, t[0], t[1], t[2],
                                                            stream_key(seed, kStreamRmat));
  TB_HIP(hipGetLastError());
}

void gen_er(tribit_ctx* ctx, uint64_t n, uint64_t nsamples, uint64_t seed, uint64_t* d_keys) {
  k_gen_er<<<gen_grid(ctx, nsamples), kBlock, 0, ctx->stream>>>(d_keys, nsamples, n, stream_key(seed, kStreamEr));
  TB_HIP(hipGetLastError());
}

// ------------------------------------------------------------- preprocessing

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

// Flags keys that are neither the sentinel nor (min < max < n).
__global__ void k_validate(const uint64_t* __restrict__ keys, uint64_t nk, uint64_t n, uint32_t* __restrict__ bad) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nk) return;
  const uint64_t k = keys[i];
  if (k == kSentinel) return;
  const uint64_t a = k >> 32, b = k & 0xFFFFFFFFull;
  if (!(a < b && b < n)) atomicOr(bad, 1u);
}

// Checks every key (min << 32) | max (min < max < n) and packs it in place to
// (min << kb) | max, so the sort covers 2 kb bits instead of 32 + kb. The
// sentinel stays all ones and still sorts last: a packed key has min < max,
// so its low 2 kb bits are never all ones.
__global__ void k_validate_pack(uint64_t* __restrict__ keys, uint64_t nk, uint64_t n, uint32_t kb,
                                uint32_t* __restrict__ bad) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nk) return;
  const uint64_t k = keys[i];
  if (k == kSentinel) return;
  const uint64_t a = k >> 32, b = k & 0xFFFFFFFFull;
  if (!(a < b && b < n)) atomicOr(bad, 1u);
  keys[i] = (a << kb) | b;
}

// pos[i] = 1 iff sorted key i is the first of its value and not the sentinel.
__global__ void k_head_flags(const uint64_t* __restrict__ k, uint64_t nk, uint32_t* __restrict__ pos) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nk) return;
  const uint64_t x = k[i];
  pos[i] = (x != kSentinel && (i == 0 || k[i - 1] != x)) ? 1u : 0u;
}

// out[pos[i]] = k[i] for the heads (pos = exclusive scan of the head flags).
__global__ void k_scatter_heads(const uint64_t* __restrict__ k, uint64_t nk, const uint32_t* __restrict__ pos,
                                uint64_t* __restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nk) return;
  if (pos[i + 1] != pos[i]) out[pos[i]] = k[i];
}

// Oriented arcs u -> v are sorted as packed keys (u << kb) | v with kb =
// bits_for(n): 2*kb bits (50 at 2^25 vertices) instead of 32 + kb, one radix
// digit pass fewer than the input key layout.
__device__ __forceinline__ uint64_t arc_key(uint32_t u, uint32_t v, uint32_t kb) {
  return ((uint64_t)u << kb) | (uint64_t)v;
}

// Degree relabelling: new id = rank of (deg, old id); lab[old] = new.
// cls[v] = floor(log2(deg[v])) + 1 (0 for an isolated vertex): octave classes.
__global__ void k_octave(const uint32_t* __restrict__ deg, uint64_t n, uint32_t* __restrict__ cls) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cls[i] = deg[i] ? 32u - (uint32_t)__clz(deg[i]) : 0u;
}

// out[i] = src[idx[i]].
__global__ void k_gather_u32(const uint32_t* __restrict__ src, const uint32_t* __restrict__ idx, uint64_t n,
                             uint32_t* __restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = src[idx[i]];
}

__global__ void k_scatter_labels(const uint32_t* __restrict__ old_of_new, uint64_t n, uint32_t* __restrict__ lab,
                                 ZeroSpans z) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  z.clear(i);
  if (i < n) lab[old_of_new[i]] = (uint32_t)i;
}

// Degree orientation: {a<b} becomes a->b iff deg(a) <= deg(b).
__global__ void k_orient(const uint64_t* __restrict__ keys, uint64_t m, const uint32_t* __restrict__ deg,
                         uint32_t kb, uint64_t* __restrict__ okeys, ZeroSpans z) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  z.clear(i);
  if (i >= m) return;
  const uint64_t k = keys[i];
  const uint32_t a = (uint32_t)(k >> kb), b = (uint32_t)(k & ((1ull << kb) - 1));
  okeys[i] = (deg[a] <= deg[b]) ? arc_key(a, b, kb) : arc_key(b, a, kb);
}

// With relabelled ids the degree order is the id order: a -> b iff a < b.
__global__ void k_orient_relabel(const uint64_t* __restrict__ keys, uint64_t m, const uint32_t* __restrict__ lab,
                                 uint32_t kb, uint64_t* __restrict__ okeys, ZeroSpans z) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  z.clear(i);
  if (i >= m) return;
  const uint64_t k = keys[i];
  const uint32_t a = lab[(uint32_t)(k >> kb)], b = lab[(uint32_t)(k & ((1ull << kb) - 1))];
  okeys[i] = a < b ? arc_key(a, b, kb) : arc_key(b, a, kb);
}

// col[i] = dst (and its low 16 bits in col16, when given: narrow wedge ranges
// are streamed from these), odeg[src] += 1 (sorted by src: aggregated per run).
__global__ void k_csr_split(const uint64_t* __restrict__ okeys, uint64_t m, uint32_t kb, uint32_t* __restrict__ col,
                            uint16_t* __restrict__ col16, uint32_t* __restrict__ odeg) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < m;
  const uint64_t k = valid ? okeys[i] : 0;
  const uint32_t s = valid ? (uint32_t)(k >> kb) : 0xFFFFFFFFu;
  if (valid) {
    const uint32_t v = (uint32_t)(k & ((1ull << kb) - 1));
    col[i] = v;
    if (col16) col16[i] = (uint16_t)v;
  } else if (col16 && i < col16_ids(m)) {
    col16[i] = 0;  // the padding to whole dwords plus one
  }
  const uint32_t run = wave_run_length(s, valid);
  if (run) atomicAdd(&odeg[s], run);
}

struct RowStats {
  unsigned long long wplus;
  unsigned long long rows_active;
  unsigned int max_outdeg;
  unsigned int row_overflow;           // build_rows' flag
  unsigned long long core_wedges[16];  // tribit_graph.core_wedges
};

// Totals over a bounded grid (grid-stride loops, one atomic per block and
// field): one atomic per wave on a single address serialises at about 13 ns
// each, 7 ms for 2^25 rows and 100 ms for 2^29 arcs.
constexpr unsigned kTotalsBlocks = 2048;
inline unsigned totals_grid(uint64_t n) {
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(kTotalsBlocks, (n + kBlock - 1) / kBlock));
}

// Edges {a, b}, a < b, of the deduplicated keys (a << kb) | b that join ids
// less than kBandIds apart, summed into *out: two keys per 16-byte load over a
// grid of at most kBandBlocks blocks, one atomic per block. keys is 256-byte
// aligned, as every block of the context's pool.
constexpr uint64_t kBandIds = 512;
constexpr unsigned kBandBlocks = 4096;
__global__ void __launch_bounds__(kBlock) k_band_edges(const uint64_t* __restrict__ keys, uint64_t m, uint32_t kb,
                                                       unsigned long long* __restrict__ out) {
  __shared__ unsigned long long s_part[kBlock / 64];
  const uint64_t lo = (1ull << kb) - 1;
  const ulonglong2* __restrict__ k2 = reinterpret_cast<const ulonglong2*>(keys);
  uint64_t acc = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m / 2;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const ulonglong2 k = k2[i];
    acc += ((k.x & lo) - (k.x >> kb) < kBandIds) + ((k.y & lo) - (k.y >> kb) < kBandIds);
  }
  if ((m & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
    const uint64_t k = keys[m - 1];
    acc += (k & lo) - (k >> kb) < kBandIds;
  }
  acc = wave_sum_u64(acc);
  if (lane_id() == 0) s_part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (unsigned i = 1; i < kBlock / 64; ++i) acc += s_part[i];
    if (acc) atomicAdd(out, (unsigned long long)acc);
  }
}

// pos[i] as k_head_flags, over a grid of at most kBandBlocks blocks, and the
// heads {a, b} (packed (a << kb) | b) that join ids less than kBandIds apart
// summed into *band, one atomic per block: the band count rides on the pass
// that dedup makes over the sorted keys anyway.
__global__ void __launch_bounds__(kBlock) k_head_flags_band(const uint64_t* __restrict__ k, uint64_t nk, uint32_t kb,
                                                            uint32_t* __restrict__ pos,
                                                            unsigned long long* __restrict__ band) {
  __shared__ unsigned long long s_part[kBlock / 64];
  const uint64_t lo = (1ull << kb) - 1;
  uint64_t acc = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nk; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t x = k[i];
    const bool head = x != kSentinel && (i == 0 || k[i - 1] != x);
    pos[i] = head ? 1u : 0u;
    acc += head && (x & lo) - (x >> kb) < kBandIds;
  }
  acc = wave_sum_u64(acc);
  if (lane_id() == 0) s_part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (unsigned i = 1; i < kBlock / 64; ++i) acc += s_part[i];
    if (acc) atomicAdd(band, (unsigned long long)acc);
  }
}

// TRIBIT_OPT_RELABEL 3 (auto). Octave-class ids keep runs of consecutive input
// ids together, which dense diagonal blocks need; degree-rank ids stream a few
// percent faster on everything else. Octave classes are taken when the edges
// joining ids less than kBandIds apart fill at least 1/16 of such id pairs:
// a block model with 512-id blocks at p_in 0.3 fills 15% of them, one at
// p_in 0.05 2.5%, a cell-ordered 2-D geometric graph of average degree 24
// 1.3%, R-MAT, Chung-Lu and Erdős–Rényi ids under 0.1%.
constexpr uint64_t kAutoMinIds = 4096;
int auto_relabel(uint64_t n, uint64_t band_edges) {
  if (n < kAutoMinIds) return 1;
  const double w = (double)std::min<uint64_t>(kBandIds, n);
  const double pairs = (w - 1.0) * (double)n - w * (w - 1.0) / 2.0;  // id pairs 1..w-1 apart
  return (double)band_edges * 16.0 >= pairs ? 2 : 1;
}

// Rows with outdeg >= 2, the largest outdeg and, with deg (undirected
// degrees), W+ = sum over v of indeg(v) * outdeg(v): every arc u -> v streams
// N+(v) once, and v has deg(v) - outdeg(v) in-arcs. With split (relabelled
// graphs), also per row the position where its last 64K-id window begins (the
// first id whose high 16 bits equal the last id's), for the narrow records of its
// wedge ranges: one lower-bound search per row. With wedges, the top ids' wedges
// by steps of kCoreStep ids, from which the core size is chosen.
__global__ void __launch_bounds__(kBlock) k_rows(const uint32_t* __restrict__ row_ptr,
                                                 const uint32_t* __restrict__ deg, const uint32_t* __restrict__ col,
                                                 uint64_t n, RowStats* __restrict__ st, uint32_t* __restrict__ split,
                                                 bool wedges) {
  __shared__ unsigned long long s_act[kBlock / 64], s_w[kBlock / 64];
  __shared__ uint32_t s_max[kBlock / 64];
  uint64_t act = 0, w = 0;
  uint32_t dm = 0;
  for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < n; u += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t b = row_ptr[u], e = row_ptr[u + 1], d = e - b;
    // wedges of the top ids: a wave's rows are neighbours, of one step or two
    if (wedges && n - u <= 16 * kCoreStep) {
      const uint32_t k = (uint32_t)((n - 1 - u) / kCoreStep);
      const uint64_t c = (uint64_t)d * (d ? d - 1 : 0) / 2, live = __ballot(true);
      const uint32_t k0 = __builtin_amdgcn_readfirstlane(k);
      if (__ballot(k == k0) == live && live == ~0ull) {
        const uint64_t sum = wave_sum_u64(c);
        if (lane_id() == 0 && sum) atomicAdd(&st->core_wedges[k], (unsigned long long)sum);
      } else if (c) {
        atomicAdd(&st->core_wedges[k], (unsigned long long)c);
      }
    }
    act += d >= 2;
    dm = d > dm ? d : dm;
    if (deg) w += (uint64_t)(deg[u] - d) * d;
    if (!split) continue;
    uint32_t lo = b;
    if (b < e) {
      const uint32_t l = col[e - 1] >> 16;
      uint32_t hi = e - 1;  // col[hi] is in window l
      while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if ((col[mid] >> 16) >= l)
          hi = mid;
        else
          lo = mid + 1;
      }
    }
    split[u] = lo;
  }
  act = wave_sum_u64(act);
  w = wave_sum_u64(w);
  dm = wave_max_u32(dm);
  if (lane_id() == 0) {
    s_act[threadIdx.x >> 6] = act;
    s_w[threadIdx.x >> 6] = w;
    s_max[threadIdx.x >> 6] = dm;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (unsigned i = 1; i < kBlock / 64; ++i) {
      act += s_act[i];
      w += s_w[i];
      dm = s_max[i] > dm ? s_max[i] : dm;
    }
    if (act) atomicAdd(&st->rows_active, (unsigned long long)act);
    if (w) atomicAdd(&st->wplus, (unsigned long long)w);
    if (dm) atomicMax(&st->max_outdeg, dm);
  }
}

// The record of arc e = (u -> v) of a relabelled graph, packed k = (u << kb) | v,
// in CSR order:
//   .x = row_ptr[u + 1] (the end of arc e's wedge range [e + 1, end), the part
//        of N+(u) after v), with bits 31 / 30 of the narrow record;
//   .y (with nar, m < 2^30) = the rest of that range's narrow record: bit 31
//        of .x: its ids share their high 16 bits H; bit 30 (with 31): shorter
//        than 2^16 ids with high halves H then H + 1, .y bits 0..15 the offset
//        of the first id with H + 1 (from the row's split position); .y bits
//        16..23 H - (v >> 16), 255 when larger. In CSR order the range's ids
//        are the row's next ones, so the reads stay in cache.
__device__ __forceinline__ uint2 arc_record(uint64_t k, uint64_t e, uint32_t kb, const uint32_t* __restrict__ row_ptr,
                                            const uint32_t* __restrict__ col, const uint32_t* __restrict__ rsplit,
                                            bool nar) {
  const uint32_t u = (uint32_t)(k >> kb);
  const uint32_t v = (uint32_t)(k & ((1ull << kb) - 1));
  const uint32_t end = row_ptr[u + 1];
  uint32_t x = end, y = 0;
  const uint32_t b = (uint32_t)e + 1;
  if (nar && b < end) {
    const uint32_t f = col[b] >> 16, l = col[end - 1] >> 16;
    const bool two = l == f + 1 && end - b < 65536u;
    if (f == l || two) {
      uint32_t d = f - (v >> 16);  // ids after v: H >= v's high half
      d = d < 255u ? d : 255u;
      x |= 0x80000000u | (two ? 0x40000000u : 0u);
      y = (d << 16) | (two ? rsplit[u] - b : 0u);
    }
  }
  return make_uint2(x, y);
}

// One 8-byte record per arc, so the wedge-range fill gathers once per range
// (graphs whose records do not fit ArcPack).
__global__ void k_arc_rec(const uint64_t* __restrict__ okeys, uint64_t m, uint32_t kb,
                          const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col,
                          const uint32_t* __restrict__ rsplit, bool nar, uint2* __restrict__ arec) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < m) arec[e] = arc_record(okeys[e], e, kb, row_ptr, col, rsplit, nar);
}

// An arc and its record in the value of the sort by head and the bits of its
// 32-bit key above the head: from bit 0, the arc (eb bits), its range's length
// (lb bits: no outdegree has more) and, with narrow records, their two flags, dh
// (8 bits) and the split offset (lb bits, below the length); the key takes what
// passes 64 bits. The sort then delivers the records in place: sorting arc
// numbers and gathering 8-byte records by them pulled a sector from HBM for each
// (R-MAT scale 25: sort 11.2 + gather 11.9 ms; with the records in the values 13.3
// + 2.7).
struct ArcPack {
  uint32_t kb, eb, lb;
  bool nar;
  __host__ __device__ uint32_t bits() const { return eb + lb + (nar ? 10 + lb : 0); }
  __host__ __device__ bool fits() const { return bits() <= 64 + (32 - kb); }
};

__global__ void k_arc_pack(const uint64_t* __restrict__ okeys, uint64_t m, ArcPack p,
                           const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col,
                           const uint32_t* __restrict__ rsplit, uint32_t* __restrict__ key,
                           uint64_t* __restrict__ val) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  const uint64_t k = okeys[e];
  const uint2 r = arc_record(k, e, p.kb, row_ptr, col, rsplit, p.nar);
  const uint32_t len = (p.nar ? r.x & 0x3FFFFFFFu : r.x) - (uint32_t)e - 1;
  unsigned __int128 w = e | ((unsigned __int128)len << p.eb);
  if (p.nar) {
    const uint64_t n = (r.x >> 30) | ((uint64_t)(r.y >> 16) << 2) | ((uint64_t)(r.y & 0xFFFFu) << 10);
    w |= (unsigned __int128)n << (p.eb + p.lb);
  }
  val[e] = (uint64_t)w;
  const uint32_t hi = (uint32_t)(w >> 64);  // zero when p.kb == 32
  key[e] = (uint32_t)(k & ((1ull << p.kb) - 1)) | (p.kb < 32 ? hi << p.kb : 0u);
}

// ------------------------------------------------------------ range lists
// For every oriented edge u->v the count streams one list: N+(v) against the
// set N+(u) ("forward", owner u) or N+(u) against the set N+(v) ("reverse",
// owner v). The streamed list is stored as its [begin, end) range in col, so
// the counting kernels read 8 coalesced bytes per edge instead of gathering
// row_ptr. Two layouts are built:
//   rng_all: all edges forward, in CSR order (owner u, row_ptr offsets);
//   rng_dir: an edge is reverse iff outdeg(u) < outdeg(v) (the shorter list
//            is streamed): forward edges per owner first (fw_ptr), then the
//            reverse edges grouped by owner v (rv_ptr, offsets past m_fwd).

__global__ void k_ranges_all(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col, uint64_t m,
                             uint2* __restrict__ rng) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m) return;
  const uint32_t v = col[e];
  rng[e] = make_uint2(row_ptr[v], row_ptr[v + 1]);
}

// Per row u: forward-edge count and forward work; reverse-edge count.
__global__ void k_dir_count(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col, uint64_t n,
                            uint32_t* __restrict__ fw_cnt, uint32_t* __restrict__ rv_out, uint64_t* __restrict__ w_fw) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u > n) return;
  uint32_t f = 0, r = 0;
  uint64_t w = 0;
  if (u < n) {
    const uint32_t r0 = row_ptr[u], r1 = row_ptr[u + 1], du = r1 - r0;
    for (uint32_t e = r0; e < r1; ++e) {
      const uint32_t v = col[e];
      const uint32_t dv = row_ptr[v + 1] - row_ptr[v];
      if (du < dv) {
        ++r;
      } else {
        ++f;
        w += dv;
      }
    }
    w_fw[u] = w;
  }
  fw_cnt[u] = f;
  rv_out[u] = r;
}

// Writes the forward ranges (and partner ids) of row u at fw_ptr[u] and its
// reverse keys (v << 32 | u) at rv_off[u].
__global__ void k_dir_fill(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col, uint64_t n,
                           const uint32_t* __restrict__ fw_ptr, const uint32_t* __restrict__ rv_off,
                           uint2* __restrict__ rng, uint32_t* __restrict__ pid, uint64_t* __restrict__ rv_keys) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  const uint32_t r0 = row_ptr[u], r1 = row_ptr[u + 1], du = r1 - r0;
  uint32_t f = fw_ptr[u], r = rv_off[u];
  for (uint32_t e = r0; e < r1; ++e) {
    const uint32_t v = col[e];
    const uint32_t b = row_ptr[v], en = row_ptr[v + 1];
    if (du < en - b) {
      rv_keys[r++] = ((uint64_t)v << 32) | (uint64_t)u;
    } else {
      pid[f] = v;
      rng[f++] = make_uint2(b, en);
    }
  }
}

// Sorted reverse keys (v << 32 | u): range of N+(u) at rng[base + j];
// rv_cnt[v] += 1 and w_rv[v] += outdeg(u), aggregated per run of v in a wave.
__global__ void k_rv_fill(const uint64_t* __restrict__ keys, uint64_t mr, const uint32_t* __restrict__ row_ptr,
                          uint2* __restrict__ rng, uint32_t* __restrict__ pid, uint32_t* __restrict__ rv_cnt,
                          unsigned long long* __restrict__ w_rv) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = j < mr;
  const uint64_t k = valid ? keys[j] : 0;
  const uint32_t v = valid ? (uint32_t)(k >> 32) : 0xFFFFFFFFu;
  uint64_t du = 0;
  if (valid) {
    const uint32_t u = (uint32_t)k;
    const uint32_t b = row_ptr[u], e = row_ptr[u + 1];
    rng[j] = make_uint2(b, e);
    pid[j] = u;
    du = e - b;
  }
  const uint32_t lane = lane_id();
  // segmented inclusive sum of du over equal v (keys sorted: equal v are contiguous)
  uint64_t sum = du;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t t = __shfl_up(sum, o);
    const uint32_t kv = __shfl_up(v, o);
    if (lane >= (uint32_t)o && kv == v) sum += t;
  }
  const uint32_t nv = __shfl_down(v, 1);
  const uint64_t vmask = __ballot(valid);
  const uint64_t above = (lane == 63) ? 0ull : (vmask >> (lane + 1));
  const bool last_valid = !(above & 1ull);
  const bool tail = valid && (last_valid || nv != v);
  const uint32_t run = wave_run_length(v, valid);
  if (run) atomicAdd(&rv_cnt[v], run);
  if (tail && sum) atomicAdd(&w_rv[v], (unsigned long long)sum);
}

// Arcs e = (u -> v) sorted by head v: the suffix of N+(u) after v,
// [e + 1, end), is streamed against N+(v). With ids in degree-rank order
// N+(v) holds only ids > v, so the elements of N+(u) up to v can never match.
// w_sfx[v] += suffix length, aggregated per run of v in a wave.
// With narrow records (arec of k_arc_rec), wedge range j = [b, e) is flagged
// narrow when its ids share their high 16 bits H (end bit 31), or, shorter
// than 2^16 ids, when they have high half H up to position b + split[j] and
// H + 1 from there (end bits 31 and 30); dh[j] = H - (v >> 16) (255: not
// representable, the counting kernel reads col[b] instead).
__global__ void k_sfx_fill(const uint32_t* __restrict__ head, const uint32_t* __restrict__ arc, uint64_t m,
                           const uint2* __restrict__ arec, uint2* __restrict__ rng, uint8_t* __restrict__ dh,
                           uint16_t* __restrict__ split, unsigned long long* __restrict__ w_sfx) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = j < m;
  const uint32_t v = valid ? head[j] : 0xFFFFFFFFu;
  uint64_t len = 0;
  if (valid) {
    const uint32_t e = arc[j];
    const uint2 r = arec[e];
    if (dh) {
      dh[j] = (uint8_t)(r.y >> 16);
      split[j] = (uint16_t)r.y;
    }
    rng[j] = make_uint2(e + 1, r.x);
    len = (r.x & 0x3FFFFFFFu) - e - 1;
  }
  uint64_t sum = 0;
  if (wave_segment_tail(v, valid, len, &sum) && sum) atomicAdd(&w_sfx[v], (unsigned long long)sum);
}

// k_sfx_fill from packed records (ArcPack) sorted by head: everything streams. A
// wave takes kUnpackSteps x 64 consecutive arcs and stores the sum of a head whose
// arcs it holds all of; only runs that may go on in another wave are added with
// atomics, which bound this pass with 64 arcs per wave: 523M arcs 5.2 ms, now 2.7
// (12 GB, 4.4 TB/s, the rate of a copy).
constexpr uint32_t kUnpackSteps = 4;
__global__ void __launch_bounds__(kBlock) k_sfx_unpack(const uint32_t* __restrict__ key,
                                                       const uint64_t* __restrict__ val, uint64_t m, ArcPack p,
                                                       uint2* __restrict__ rng, uint8_t* __restrict__ dh,
                                                       uint16_t* __restrict__ split,
                                                       unsigned long long* __restrict__ w_sfx) {
  const uint32_t lane = lane_id();
  const uint64_t j0 = ((uint64_t)blockIdx.x * kBlock + (threadIdx.x & ~63u)) * kUnpackSteps + lane;
  uint32_t k[kUnpackSteps];
  uint64_t lo[kUnpackSteps];
#pragma unroll
  for (uint32_t t = 0; t < kUnpackSteps; ++t) {
    const uint64_t j = j0 + 64 * t;
    k[t] = j < m ? key[j] : 0u;
    lo[t] = j < m ? val[j] : 0ull;
  }
  bool carried = false, open = true;  // a run of the last step goes on; it reaches back to the wave's first arc
  uint32_t ck = 0, cs = 0;            // its head and sum
#pragma unroll
  for (uint32_t t = 0; t < kUnpackSteps; ++t) {
    const uint64_t j = j0 + 64 * t;
    const bool valid = j < m;
    const uint32_t v = valid ? (uint32_t)(k[t] & ((1ull << p.kb) - 1)) : 0xFFFFFFFFu;
    uint32_t len = 0;
    if (valid) {
      const unsigned __int128 w = ((unsigned __int128)(p.kb < 32 ? k[t] >> p.kb : 0u) << 64) | lo[t];
      const uint32_t b = (uint32_t)((uint64_t)w & ((1ull << p.eb) - 1)) + 1;
      len = (uint32_t)((uint64_t)(w >> p.eb) & ((1ull << p.lb) - 1));
      uint32_t x = b + len;
      if (p.nar) {
        const uint64_t n = (uint64_t)(w >> (p.eb + p.lb));
        x |= (uint32_t)(n & 3) << 30;
        dh[j] = (uint8_t)(n >> 2);
        split[j] = (uint16_t)((n >> 10) & ((1ull << p.lb) - 1));
      }
      rng[j] = make_uint2(b, x);
    }
    uint32_t sum = 0;  // 64 kUnpackSteps lengths of at most 2^17
    const bool tail = wave_segment_tail_u32(v, valid, len, &sum);
    const uint32_t v0 = __shfl(v, 0), v63 = __shfl(v, 63);
    const bool full = __shfl((int)valid, 63), joins = carried && ck == v0;
    if (carried && !joins && lane == 0 && cs) {  // the run ended with the last step
      if (open)
        atomicAdd(&w_sfx[ck], (unsigned long long)cs);
      else
        w_sfx[ck] = cs;
    }
    const bool reaches = t == 0 || (joins && open);  // this step's first run: back to the wave's first arc
    if (joins && v == v0) sum += cs;
    const bool last = full && v == v63;
    if (tail && sum && !(last && t + 1 < kUnpackSteps)) {
      if (last || (reaches && v == v0))
        atomicAdd(&w_sfx[v], (unsigned long long)sum);
      else
        w_sfx[v] = sum;
    }
    carried = full;
    open = reaches && v63 == v0;
    ck = v63;
    cs = __shfl(sum, 63);
  }
}

// W+(u) = sum of outdeg(v) over v in N+(u), per row (the PLAIN layout's work).
__global__ void k_row_wplus(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col, uint64_t n,
                            uint64_t* __restrict__ wrow) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  uint64_t w = 0;
  for (uint32_t e = row_ptr[u]; e < row_ptr[u + 1]; ++e) {
    const uint32_t v = col[e];
    w += row_ptr[v + 1] - row_ptr[v];
  }
  wrow[u] = w;
}

__global__ void k_fill_u64(unsigned long long* __restrict__ p, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0ull;
}

__global__ void k_add_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] += v;
}

// Sorts and scans of at most kSmallSort items: one workgroup, one launch. The
// device-wide ones are seven or eight launches at these sizes (a block sort and
// its merge steps), about 7 us each, and most of what a small graph's
// preprocessing took: 1,000 vertices and 8,000 keys 0.35 -> 0.2 ms a call, with
// the passes over n and m that now share a launch.
constexpr uint32_t kSmallSort = 8192;
constexpr uint32_t kSmallThreads = 1024;
constexpr uint32_t kSmallItems = kSmallSort / kSmallThreads;

// Missing items get the largest key of `bits` bits and, the sort being stable, stay last.
template <typename K, typename V>
__global__ void __launch_bounds__(kSmallThreads) k_sort_small(const K* __restrict__ in, K* __restrict__ out,
                                                              const V* __restrict__ vin, V* __restrict__ vout,
                                                              uint32_t n, uint32_t bits) {
  using Sort = rocprim::block_radix_sort<K, kSmallThreads, kSmallItems, V>;
  __shared__ typename Sort::storage_type tmp;
  K k[kSmallItems];
  V v[kSmallItems];
#pragma unroll
  for (uint32_t j = 0; j < kSmallItems; ++j) {
    const uint32_t i = threadIdx.x * kSmallItems + j;
    k[j] = i < n ? in[i] : (K)~(K)0;
    v[j] = i < n ? (vin ? vin[i] : (V)i) : (V)0;
  }
  Sort().sort_to_striped(k, v, tmp, 0, bits);
#pragma unroll
  for (uint32_t j = 0; j < kSmallItems; ++j) {
    const uint32_t i = threadIdx.x + j * kSmallThreads;
    if (i < n) {
      out[i] = k[j];
      vout[i] = v[j];
    }
  }
}

__global__ void __launch_bounds__(kSmallThreads) k_sort_small_keys(const uint64_t* __restrict__ in,
                                                                   uint64_t* __restrict__ out, uint32_t n,
                                                                   uint32_t bits) {
  using Sort = rocprim::block_radix_sort<uint64_t, kSmallThreads, kSmallItems>;
  __shared__ typename Sort::storage_type tmp;
  uint64_t k[kSmallItems];
#pragma unroll
  for (uint32_t j = 0; j < kSmallItems; ++j) {
    const uint32_t i = threadIdx.x * kSmallItems + j;
    k[j] = i < n ? in[i] : ~0ull;
  }
  Sort().sort_to_striped(k, tmp, 0, bits);
#pragma unroll
  for (uint32_t j = 0; j < kSmallItems; ++j) {
    const uint32_t i = threadIdx.x + j * kSmallThreads;
    if (i < n) out[i] = k[j];
  }
}

// The sorted keys' numbers, or the values vin, into vout.
static void sort_pairs(tribit_ctx* ctx, const uint32_t* in, uint32_t* out, uint32_t* order, uint64_t n, uint32_t bits) {
  if (n <= kSmallSort)
    k_sort_small<uint32_t, uint32_t><<<1, kSmallThreads, 0, ctx->stream>>>(in, out, nullptr, order, (uint32_t)n, bits);
  else
    sort_ids_device(ctx, in, out, order, n, bits);
}
static void sort_pairs(tribit_ctx* ctx, const uint32_t* in, uint32_t* out, const uint64_t* vin, uint64_t* vout,
                       uint64_t n, uint32_t bits) {
  if (n <= kSmallSort)
    k_sort_small<uint32_t, uint64_t><<<1, kSmallThreads, 0, ctx->stream>>>(in, out, vin, vout, (uint32_t)n, bits);
  else
    sort_records_device(ctx, in, out, vin, vout, n, bits);
}

struct InDegree {
  const uint32_t *deg, *odeg;
  uint64_t n;
  __host__ __device__ uint32_t operator()(uint64_t v) const { return v < n ? deg[v] - odeg[v] : 0u; }
};

struct OutDegree {
  const uint32_t* odeg;
  __device__ uint32_t operator()(uint64_t v) const { return odeg[v]; }
};

// Both scans of scan_rows for small n: a workgroup each in one launch.
__global__ void __launch_bounds__(kScanBlockThreads) k_scan_small(OutDegree f, InDegree g, uint32_t n,
                                                                  uint32_t* __restrict__ row_ptr,
                                                                  uint32_t* __restrict__ sfx_ptr) {
  if (blockIdx.x == 0)
    scan_block(f, n, row_ptr);
  else
    scan_block(g, n, sfx_ptr);
}

// out[0, n): the exclusive scan of in (every caller through one instance of the device-wide scan).
static void scan_u32(tribit_ctx* ctx, const uint32_t* in, uint32_t* out, uint64_t n) {
  with_temp(ctx, [&](void* t, size_t& b) {
    return rocprim::exclusive_scan(t, b, in, out, 0u, (size_t)n, rocprim::plus<uint32_t>(), ctx->stream);
  });
}

// row_ptr[n + 1], the exclusive scan of odeg[0, n], and, with sfx_ptr, that of the
// in-degrees deg - odeg.
static void scan_rows(tribit_ctx* ctx, const uint32_t* odeg, const uint32_t* deg, uint64_t n, uint32_t* row_ptr,
                      uint32_t* sfx_ptr) {
  hipStream_t s = ctx->stream;
  if (n <= kSmallScan) {
    k_scan_small<<<sfx_ptr ? 2 : 1, kScanBlockThreads, 0, s>>>(OutDegree{odeg}, InDegree{deg, odeg, n}, (uint32_t)n,
                                                              row_ptr, sfx_ptr);
    return;
  }
  scan_u32(ctx, odeg, row_ptr, n + 1);
  if (!sfx_ptr) return;
  const auto indeg = rocprim::make_transform_iterator(rocprim::counting_iterator<uint64_t>(0), InDegree{deg, odeg, n});
  with_temp(ctx, [&](void* t, size_t& b) {
    return rocprim::exclusive_scan(t, b, indeg, sfx_ptr, 0u, (size_t)(n + 1), rocprim::plus<uint32_t>(), s);
  });
}

static void sort_keys(tribit_ctx* ctx, const uint64_t* in, uint64_t* out, uint64_t nk, uint32_t end_bit) {
  if (nk <= kSmallSort) {
    if (nk) k_sort_small_keys<<<1, kSmallThreads, 0, ctx->stream>>>(in, out, (uint32_t)nk, end_bit);
    return;
  }
  sort_keys_device(ctx, in, out, nk, end_bit);
}

// Where the labels of kSkewIds ids or more begin in their buffer (in ids): an
// R-MAT graph's frequent endpoints are ids with few set bits, and the label
// gathers of k_row_split met in few memory channels when the array began at a
// multiple of 2 MiB (scale 25: 13.6 ms; 12.0 from 1 MiB past one; 11.0 to 11.4
// from an offset of many set bits). Smaller label arrays stay in L2.
constexpr uint64_t kSkewIds = 1ull << 20;
constexpr uint64_t kLabelSkew = 0x1D9500 / 4;

void preprocess(tribit_ctx* ctx, uint64_t* d_keys_in, uint64_t nkeys, uint64_t n, tribit_graph* g, int relabel_opt) {
  if (relabel_opt < 0) relabel_opt = ctx->relabel;
  DevBuf<uint64_t> keys;
  keys.ctx = ctx;
  keys.p = d_keys_in;  // owned from here on
  keys.n = nkeys;
  if (n == 0 || n > 0xFFFFFFFEull) fail(TRIBIT_ERR_TOO_LARGE, "vertex count must be in [1, 2^32-2]");
  hipStream_t s = ctx->stream;
  g->ctx = ctx;
  g->n = n;
  g->entries = nkeys;
  // the code that a graph of this size comes to, unless a partition overflows
  if (relabel_opt && n > kSmallSort) load_sort_ids(ctx);
  if (nkeys > kSmallSort) {
    if (relabel_opt) {
      load_rows(ctx);
      load_sort_records(ctx);
    } else {
      load_sort_keys(ctx);
    }
  }
  TB_HIP(hipEventRecord(ctx->ev[0], s));

  // keys checked and packed to (min << kb) | max for the sort
  const uint32_t kb = bits_for(n);

  // 1-2. distinct keys (tribit.cu:666-667): by partition, in any order; the
  // sort, after which the sentinel comes last, is for keys repeated so often
  // that a bucket of the partition overflows and for more than 2^32 - 2 keys.
  const uint32_t end_bit = 2 * kb;
  uint64_t m = 0;
  // id-band edges for the automatic choice of ids (TRIBIT_OPT_RELABEL 3)
  const bool want_band = relabel_opt == 3 && n >= kAutoMinIds;
  uint64_t band_edges = 0;
  DevBuf<unsigned long long> band;
  band.ctx = ctx;
  DevBuf<uint64_t> uniq(ctx, nkeys ? nkeys : 1);
  bool bad_key = false, distinct = false;
  if (nkeys && nkeys <= 0xFFFFFFFEull) {
    try {
      distinct = distinct_keys(ctx, keys.p, nkeys, n, kb, uniq.p, &m, &bad_key, kBandIds,
                               want_band ? &band_edges : nullptr);
    } catch (const Error& e) {  // the partition's regions take more room than the sort's
      if (e.status != TRIBIT_ERR_NOMEM) throw;
    }
  }
  if (distinct) {
    keys.reset();
    if (bad_key) fail(TRIBIT_ERR_RANGE, "edge key is not (min < max < n)");
  } else if (nkeys) {
    DevBuf<uint32_t> flag(ctx, 4);
    k_fill_u32<<<1, 64, 0, s>>>(flag.p, 4, 0u);
    k_validate_pack<<<grid_for(nkeys, kBlock), kBlock, 0, s>>>(keys.p, nkeys, n, kb, flag.p);
    DevBuf<uint64_t> sorted(ctx, nkeys);
    sort_keys(ctx, keys.p, sorted.p, nkeys, end_bit);
    keys.reset();
    // unique: head flags, their exclusive scan (the last entry is the count),
    // scatter of the heads; the sentinel is never a head. 32-bit positions
    // (rocprim::unique took 16 ms for the 537M keys of R-MAT scale 25; more
    // than 2^32 - 2 keys still go through it).
    uint32_t bad = 0;
    if (nkeys <= 0xFFFFFFFEull) {
      DevBuf<uint32_t> head(ctx, nkeys + 1), pos(ctx, nkeys + 1);
      if (want_band) {
        band = DevBuf<unsigned long long>(ctx, 1);
        k_fill_u32<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t*>(band.p), 2, 0u);
        const unsigned grid = (unsigned)std::min<uint64_t>(kBandBlocks, (nkeys + kBlock - 1) / kBlock);
        k_head_flags_band<<<grid, kBlock, 0, s>>>(sorted.p, nkeys, kb, head.p, band.p);
      } else {
        k_head_flags<<<grid_for(nkeys, kBlock), kBlock, 0, s>>>(sorted.p, nkeys, head.p);
      }
      k_fill_u32<<<1, 64, 0, s>>>(head.p + nkeys, 1, 0u);
      scan_u32(ctx, head.p, pos.p, nkeys + 1);
      k_scatter_heads<<<grid_for(nkeys, kBlock), kBlock, 0, s>>>(sorted.p, nkeys, pos.p, uniq.p);
      uint32_t cnt = 0;
      TB_HIP(hipMemcpyAsync(&cnt, pos.p + nkeys, 4, hipMemcpyDeviceToHost, s));
      TB_HIP(hipMemcpyAsync(&bad, flag.p, 4, hipMemcpyDeviceToHost, s));
      if (want_band) TB_HIP(hipMemcpyAsync(&band_edges, band.p, 8, hipMemcpyDeviceToHost, s));
      ctx->sync();
      band.reset();
      m = cnt;
    } else {
      DevBuf<uint64_t> ucount(ctx, 1);
      unique_device(ctx, sorted.p, uniq.p, ucount.p, nkeys);
      uint64_t h[2] = {0, 0};
      TB_HIP(hipMemcpyAsync(&h[0], ucount.p, 8, hipMemcpyDeviceToHost, s));
      ctx->sync();
      if (h[0]) TB_HIP(hipMemcpyAsync(&h[1], uniq.p + h[0] - 1, 8, hipMemcpyDeviceToHost, s));
      TB_HIP(hipMemcpyAsync(&bad, flag.p, 4, hipMemcpyDeviceToHost, s));
      ctx->sync();
      m = h[0] - ((h[0] && h[1] == kSentinel) ? 1 : 0);
      if (want_band && m && !bad) {
        band = DevBuf<unsigned long long>(ctx, 1);
        k_fill_u32<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t*>(band.p), 2, 0u);
        const unsigned grid = (unsigned)std::min<uint64_t>(kBandBlocks, (m / 2 + kBlock) / kBlock);
        k_band_edges<<<grid, kBlock, 0, s>>>(uniq.p, m, kb, band.p);
        TB_HIP(hipMemcpyAsync(&band_edges, band.p, 8, hipMemcpyDeviceToHost, s));
        ctx->sync();
        band.reset();
      }
    }
    if (bad) fail(TRIBIT_ERR_RANGE, "edge key is not (min < max < n)");
  } else {
    keys.reset();
  }
  if (m > 0xFFFFFFFFull) fail(TRIBIT_ERR_TOO_LARGE, "more than 2^32-1 edges in one graph");
  g->m = m;

  // 3. degrees
  DevBuf<uint32_t> deg(ctx, n, kKept);
  count_degrees(ctx, uniq.p, m, n, kb, deg.p);

  // 3b. optional degree relabelling: internal id = rank of (deg, id) (mode 1)
  // or of (octave of deg, id) (mode 2; mode 3 picks 1 or 2 from the id-band
  // edges), so the orientation below becomes the id order and the
  // out-neighbours of high-degree vertices are packed into a narrow id range
  // at the top.
  const int relabel = relabel_opt == 3 ? auto_relabel(n, band_edges) : relabel_opt;
  DevBuf<uint32_t> labels;
  labels.ctx = ctx;
  DevBuf<uint64_t> okeys;  // oriented arcs, packed (u << kb) | v
  okeys.ctx = ctx;
  // Buffers are taken where they are first used and given back after their last
  // use: with the fall-backs to sorts on NOMEM, a build needs no more than the
  // sorts do, max(32 nkeys, 43 m + 28 n) bytes (degree-rank ids).
  DevBuf<uint32_t> odeg;
  DevBuf<RowStats> st(ctx, 1);
  DevBuf<uint64_t> w_sfx;
  odeg.ctx = w_sfx.ctx = ctx;
  ZeroSpans zero{};
  const auto take_zeroed = [&] {  // odeg, st and w_sfx, cleared by the next launch
    odeg = DevBuf<uint32_t>(ctx, n + 1);
    if (relabel) w_sfx = DevBuf<uint64_t>(ctx, n, kKept);
    zero = ZeroSpans{{odeg.p, reinterpret_cast<uint32_t*>(st.p), reinterpret_cast<uint32_t*>(w_sfx.p)},
                     {n + 1, sizeof(RowStats) / 4, relabel ? 2 * n : 0}};
  };
  // 4-6. the arcs sorted by (u, v) into the CSR
  const bool narrow = relabel && m && m < (1ull << 30);
  DevBuf<uint32_t> col, col16;
  col.ctx = col16.ctx = ctx;
  const auto take_columns = [&] {
    col = DevBuf<uint32_t>(ctx, m ? m : 1, kKept);
    if (narrow) col16 = DevBuf<uint32_t>(ctx, col16_ids(m) / 2, kKept);
  };
  const auto ids16 = [&] { return reinterpret_cast<uint16_t*>(col16.p); };
  bool sorted = false;
  if (relabel) {
    labels = DevBuf<uint32_t>(ctx, n, kKept);
    {
      DevBuf<uint32_t> deg_sorted(ctx, n, kKept);
      if (relabel == 2) {
        // octave classes: rank of (floor(log2(deg)), id); runs of consecutive
        // input ids with similar degrees (a block of a block model) stay runs
        DevBuf<uint32_t> cls(ctx, n);
        k_octave<<<grid_for(n, kBlock), kBlock, 0, s>>>(deg.p, n, cls.p);
        sort_pairs(ctx, cls.p, deg_sorted.p, labels.p, n, 6u);
        k_gather_u32<<<grid_for(n, kBlock), kBlock, 0, s>>>(deg.p, labels.p, n, deg_sorted.p);
      } else {
        sort_pairs(ctx, deg.p, deg_sorted.p, labels.p, n, bits_for(n));
      }
      std::swap(deg.p, deg_sorted.p);  // deg now indexed by internal id
    }
    const uint64_t skew = n >= kSkewIds ? kLabelSkew : 0;
    DevBuf<uint32_t> lab_buf(ctx, n + skew);
    uint32_t* lab = lab_buf.p + skew;
    take_zeroed();
    const unsigned grid = grid_for(zero.grid_items(n), kBlock);
    k_scatter_labels<<<grid, kBlock, 0, s>>>(labels.p, n, lab, zero);
    take_columns();
    // rows by partition, but a sort by one workgroup where that suffices (two
    // launches of 35 us against five of 31) and for more edges than the slots cover
    if (m > kSmallSort && m < kRowsMaxEdges) {
      try {
        build_rows(ctx, uniq.p, m, lab, deg.p, n, kb, uniq.p, col.p, ids16(), odeg.p, &st.p->row_overflow);
        sorted = true;
      } catch (const Error& e) {  // the slots take more room than the sort
        if (e.status != TRIBIT_ERR_NOMEM) throw;
      }
    }
    if (m && !sorted) {
      okeys = DevBuf<uint64_t>(ctx, m);
      k_orient_relabel<<<grid_for(m, kBlock), kBlock, 0, s>>>(uniq.p, m, lab, kb, okeys.p, ZeroSpans{});
    }
  } else {
    if (m) okeys = DevBuf<uint64_t>(ctx, m);
    take_zeroed();
    const unsigned grid = grid_for(zero.grid_items(m), kBlock);
    k_orient<<<grid, kBlock, 0, s>>>(uniq.p, m, deg.p, kb, okeys.p, zero);
    take_columns();
  }
  if (m && !sorted) {
    sort_keys(ctx, okeys.p, uniq.p, m, 2 * kb);
    okeys.reset();
    k_csr_split<<<grid_for(m + 4, kBlock), kBlock, 0, s>>>(uniq.p, m, kb, col.p, ids16(), odeg.p);
  }
  DevBuf<uint32_t> row_ptr(ctx, n + 1, kKept);
  DevBuf<uint32_t> sfx_ptr;
  sfx_ptr.ctx = ctx;
  if (relabel) sfx_ptr = DevBuf<uint32_t>(ctx, n + 1, kKept);
  scan_rows(ctx, odeg.p, deg.p, n, row_ptr.p, sfx_ptr.p);
  odeg.reset();

  // 7. totals (W+, active rows, largest outdeg) from the rows, and the rows' split positions
  DevBuf<uint32_t> rsplit;
  rsplit.ctx = ctx;
  if (narrow) rsplit = DevBuf<uint32_t>(ctx, n);
  k_rows<<<totals_grid(n), kBlock, 0, s>>>(row_ptr.p, deg.p, col.p, n, st.p, rsplit.p, relabel != 0);
  RowStats hst;

  // 8. wedge ranges (relabelled graphs): in-arcs of every v, each with its
  // suffix range; narrow ranges flagged (streamed from col16)
  DevBuf<uint2> rng_sfx;
  DevBuf<uint8_t> sfx_dh;
  DevBuf<uint16_t> sfx_split;
  rng_sfx.ctx = ctx;
  if (relabel) {
    rng_sfx = DevBuf<uint2>(ctx, m ? m : 1, kKept);
    if (narrow) {
      sfx_dh = DevBuf<uint8_t>(ctx, m, kKept);
      sfx_split = DevBuf<uint16_t>(ctx, m, kKept);
    }
    if (m) {
      // no outdegree passes 2 sqrt(m): its vertices' degrees (octave ids: half of
      // them) are all at least as large. The real largest is asked for only when
      // that bound leaves the records too wide.
      ArcPack pack{kb, bits_for(m), bits_for((uint64_t)(2.0 * std::sqrt((double)m)) + 2), narrow};
      if (!pack.fits()) {
        TB_HIP(hipMemcpyAsync(&hst, st.p, sizeof(hst), hipMemcpyDeviceToHost, s));
        ctx->sync();
        pack.lb = bits_for((uint64_t)hst.max_outdeg + 1);
      }
      unsigned long long* w = reinterpret_cast<unsigned long long*>(w_sfx.p);
      bool filled = false;
      if (pack.fits()) {
        try {
          DevBuf<uint32_t> key(ctx, m), key_sorted(ctx, m);
          DevBuf<uint64_t> val(ctx, m), val_sorted(ctx, m);
          k_arc_pack<<<grid_for(m, kBlock), kBlock, 0, s>>>(uniq.p, m, pack, row_ptr.p, col.p, rsplit.p, key.p, val.p);
          sort_pairs(ctx, key.p, key_sorted.p, val.p, val_sorted.p, m, kb);
          k_sfx_unpack<<<grid_for(m, kBlock * kUnpackSteps), kBlock, 0, s>>>(
              key_sorted.p, val_sorted.p, m, pack, rng_sfx.p, sfx_dh.p, sfx_split.p, w);
          filled = true;
        } catch (const Error& e) {  // 36 bytes an arc beside the keys; arc numbers and records take 24 without them
          if (e.status != TRIBIT_ERR_NOMEM) throw;
        }
      }
      if (!filled) {
        DevBuf<uint2> arec(ctx, m);
        k_arc_rec<<<grid_for(m, kBlock), kBlock, 0, s>>>(uniq.p, m, kb, row_ptr.p, col.p, rsplit.p, narrow, arec.p);
        uniq.reset();
        rsplit.reset();
        DevBuf<uint32_t> head(ctx, m), arc_sorted(ctx, m);
        sort_pairs(ctx, col.p, head.p, arc_sorted.p, m, kb);
        k_sfx_fill<<<grid_for(m, kBlock), kBlock, 0, s>>>(head.p, arc_sorted.p, m, arec.p, rng_sfx.p, sfx_dh.p,
                                                          sfx_split.p, w);
      }
    }
  }
  rsplit.reset();
  uniq.reset();
  TB_HIP(hipMemcpyAsync(&hst, st.p, sizeof(hst), hipMemcpyDeviceToHost, s));

  // the graph owns its buffers from here on (freed by tribit_graph_free, also on error)
  g->row_ptr = row_ptr.release();
  g->col = col.release();
  g->deg = deg.release();
  g->labels = labels.release();
  g->relabeled = relabel;
  g->rng_sfx = rng_sfx.release();
  g->col16 = reinterpret_cast<uint16_t*>(col16.release());
  g->sfx_dh = sfx_dh.release();
  g->sfx_split = sfx_split.release();
  g->sfx_ptr = sfx_ptr.release();
  g->w_sfx = w_sfx.release();
  g->bytes = 4 * (n + 1) + 4 * (m ? m : 1) + 4 * n + (g->labels ? 4 * n : 0) +
             (g->rng_sfx ? 8 * (m ? m : 1) + 4 * (n + 1) + 8 * n : 0) + (g->col16 ? 4 * ((m + 1) / 2 + 1) + 3 * m : 0);
  // a graph without wedge ranges counts on the direction-split layout by default: built here
  if (!g->rng_sfx) build_layout(ctx, g, TRIBIT_SCHED_DIRECTED);
  TB_HIP(hipEventRecord(ctx->ev[1], s));
  TB_HIP(hipEventSynchronize(ctx->ev[1]));
  TB_HIP(hipGetLastError());
  float ms = 0.f;
  TB_HIP(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
  g->ms_prep = ms;
  if (hst.row_overflow) fail(TRIBIT_ERR_HIP, "a row passed its degree bound");
  g->wplus = hst.wplus;
  g->rows_active = hst.rows_active;
  g->max_outdeg = hst.max_outdeg;
  for (int k = 0; k < 16; ++k) g->core_wedges[k] = hst.core_wedges[k];
}

// ------------------------------------------------------------ range layouts
// The layouts a schedule streams beside the wedge ranges: rng_all (PLAIN,
// every arc forward in CSR order) and rng_dir (DIRECTED). Preprocessing builds
// the graph's default one (wedge ranges for relabelled graphs, else DIRECTED);
// the others are built on their first use, outside the count's timing, and
// their device time is kept per layout (tribit_graph_info.ms_layout).
void build_layout(tribit_ctx* ctx, tribit_graph* g, int layout) {
  hipStream_t s = ctx->stream;
  const uint64_t n = g->n, m = g->m;
  if (layout == TRIBIT_SCHED_PLAIN) {
    DevBuf<uint2> rng_all(ctx, m ? m : 1, kKept);
    DevBuf<uint64_t> wrow(ctx, n ? n : 1, kKept);
    if (m) k_ranges_all<<<grid_for(m, kBlock), kBlock, 0, s>>>(g->row_ptr, g->col, m, rng_all.p);
    if (n) k_row_wplus<<<grid_for(n, kBlock), kBlock, 0, s>>>(g->row_ptr, g->col, n, wrow.p);
    TB_HIP(hipGetLastError());
    g->rng_all = rng_all.release();
    g->wrow = wrow.release();
    g->bytes += 8 * (m ? m : 1) + 8 * (n ? n : 1);
    return;
  }
  if (layout != TRIBIT_SCHED_DIRECTED) fail(TRIBIT_ERR_ARG, "no such range layout");
  const uint32_t end_bit = 32 + bits_for(n);
  DevBuf<uint2> rng_dir(ctx, m ? m : 1, kKept);
  DevBuf<uint32_t> pid_dir(ctx, m ? m : 1, kKept);
  DevBuf<uint32_t> fw_ptr(ctx, n + 1, kKept), rv_ptr(ctx, n + 1, kKept);
  DevBuf<uint64_t> w_fw(ctx, n, kKept), w_rv(ctx, n, kKept);
  uint32_t m_fwd = 0;
  k_fill_u64<<<grid_for(n, kBlock), kBlock, 0, s>>>(reinterpret_cast<unsigned long long*>(w_rv.p), n);
  if (m) {
    DevBuf<uint32_t> fw_cnt(ctx, n + 1), rv_cnt(ctx, n + 1), rv_off(ctx, n + 1);
    k_dir_count<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(g->row_ptr, g->col, n, fw_cnt.p, rv_cnt.p, w_fw.p);
    scan_u32(ctx, fw_cnt.p, fw_ptr.p, n + 1);
    scan_u32(ctx, rv_cnt.p, rv_off.p, n + 1);
    TB_HIP(hipMemcpyAsync(&m_fwd, fw_ptr.p + n, 4, hipMemcpyDeviceToHost, s));
    ctx->sync();
    const uint64_t m_rev = m - m_fwd;
    DevBuf<uint64_t> rv_keys(ctx, m_rev ? m_rev : 1);
    k_dir_fill<<<grid_for(n, kBlock), kBlock, 0, s>>>(g->row_ptr, g->col, n, fw_ptr.p, rv_off.p, rng_dir.p,
                                                      pid_dir.p, rv_keys.p);
    k_fill_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(rv_cnt.p, n + 1, 0u);
    if (m_rev) {
      DevBuf<uint64_t> rv_sorted(ctx, m_rev);
      sort_keys(ctx, rv_keys.p, rv_sorted.p, m_rev, end_bit);
      k_rv_fill<<<grid_for(m_rev, kBlock), kBlock, 0, s>>>(rv_sorted.p, m_rev, g->row_ptr, rng_dir.p + m_fwd,
                                                           pid_dir.p + m_fwd, rv_cnt.p,
                                                           reinterpret_cast<unsigned long long*>(w_rv.p));
    }
    scan_u32(ctx, rv_cnt.p, rv_ptr.p, n + 1);
    k_add_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(rv_ptr.p, n + 1, m_fwd);
  } else {
    k_fill_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(fw_ptr.p, n + 1, 0u);
    k_fill_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(rv_ptr.p, n + 1, 0u);
    k_fill_u64<<<grid_for(n, kBlock), kBlock, 0, s>>>(reinterpret_cast<unsigned long long*>(w_fw.p), n);
  }
  TB_HIP(hipGetLastError());
  g->m_fwd = m_fwd;
  g->rng_dir = rng_dir.release();
  g->pid_dir = pid_dir.release();
  g->fw_ptr = fw_ptr.release();
  g->rv_ptr = rv_ptr.release();
  g->w_fw = w_fw.release();
  g->w_rv = w_rv.release();
  g->bytes += 12 * (m ? m : 1) + 8 * (n + 1) + 16 * n;
}

bool layout_built(const tribit_graph* g, int layout) {
  if (layout == TRIBIT_SCHED_PLAIN) return g->rng_all != nullptr;
  if (layout == TRIBIT_SCHED_DIRECTED) return g->rng_dir != nullptr;
  if (layout == TRIBIT_SCHED_WEDGE) return g->rng_sfx != nullptr;
  return false;
}

void ensure_layout(tribit_ctx* ctx, tribit_graph* g, int layout) {
  if (layout_built(g, layout)) return;
  if (layout == TRIBIT_SCHED_WEDGE) fail(TRIBIT_ERR_ARG, "wedge ranges need a relabelled graph (TRIBIT_OPT_RELABEL)");
  hipStream_t s = ctx->stream;
  hipEvent_t a = nullptr, b = nullptr;
  TB_HIP(hipEventCreate(&a));
  TB_HIP(hipEventCreate(&b));
  if (layout == TRIBIT_SCHED_DIRECTED && g->m > kSmallSort) load_sort_keys(ctx);
  TB_HIP(hipEventRecord(a, s));
  build_layout(ctx, g, layout);
  TB_HIP(hipEventRecord(b, s));
  TB_HIP(hipEventSynchronize(b));
  float ms = 0.f;
  TB_HIP(hipEventElapsedTime(&ms, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  g->ms_layout[layout] = ms;
}

// ------------------------------------------- one rank's off-diagonal task
// The reference's off-diagonal task (main6_multi.cu:595-751, task shapes
// main.rs:186-220) counts the triangles a < b < c with (a, b) in `cols` and
// (a, c), (b, c) in `idxs`. As a count of this library: the idxs edges x -> c
// (x the smaller id) form the CSR H; every cols edge {a, b} is one streamed
// list, H's row of one endpoint against the set of H's row of the other, the
// endpoint with the longer row owning the set. The lists go into the reverse
// part of a direction-split layout (no forward part), which the DIRECTED
// schedule counts unchanged.

// Owner-first keys (o << 32) | s of the cols edges: o the endpoint with the
// longer H row (ties: the larger id); sentinels stay sentinels.
__global__ void k_offdiag_keys(const uint64_t* __restrict__ keys, uint64_t nk, const uint32_t* __restrict__ hrp,
                               uint64_t* __restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nk) return;
  const uint64_t k = keys[i];
  if (k == kSentinel) {
    out[i] = kSentinel;
    return;
  }
  const uint32_t a = (uint32_t)(k >> 32), b = (uint32_t)k;
  const uint32_t la = hrp[a + 1] - hrp[a], lb = hrp[b + 1] - hrp[b];
  out[i] = la > lb ? (((uint64_t)a << 32) | b) : (((uint64_t)b << 32) | a);
}

// Sum of v[0, n) into *out (launched on totals_grid(n) blocks of kBlock).
__global__ void __launch_bounds__(kBlock) k_sum_u64(const unsigned long long* __restrict__ v, uint64_t n,
                                                    unsigned long long* __restrict__ out) {
  __shared__ unsigned long long s_part[kBlock / 64];
  uint64_t acc = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    acc += v[i];
  acc = wave_sum_u64(acc);
  if (lane_id() == 0) s_part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (unsigned i = 1; i < kBlock / 64; ++i) acc += s_part[i];
    if (acc) atomicAdd(out, (unsigned long long)acc);
  }
}

// Sorted distinct keys of in[0, nk) (the sentinel dropped) into out; returns
// their number. Sets *bad when a key is not (min < max < n).
static uint64_t sort_unique(tribit_ctx* ctx, const uint64_t* in, uint64_t nk, uint64_t n, uint64_t* out, bool* bad) {
  hipStream_t s = ctx->stream;
  if (!nk) return 0;
  if (nk > 0xFFFFFFFEull) fail(TRIBIT_ERR_TOO_LARGE, "more than 2^32-2 keys in one task set");
  DevBuf<uint32_t> flag(ctx, 1);
  k_fill_u32<<<1, 64, 0, s>>>(flag.p, 1, 0u);
  k_validate<<<grid_for(nk, kBlock), kBlock, 0, s>>>(in, nk, n, flag.p);
  DevBuf<uint64_t> sorted(ctx, nk);
  sort_keys(ctx, in, sorted.p, nk, 32 + bits_for(n));
  DevBuf<uint32_t> head(ctx, nk + 1), pos(ctx, nk + 1);
  k_head_flags<<<grid_for(nk, kBlock), kBlock, 0, s>>>(sorted.p, nk, head.p);
  k_fill_u32<<<1, 64, 0, s>>>(head.p + nk, 1, 0u);
  scan_u32(ctx, head.p, pos.p, nk + 1);
  k_scatter_heads<<<grid_for(nk, kBlock), kBlock, 0, s>>>(sorted.p, nk, pos.p, out);
  uint32_t cnt = 0, f = 0;
  TB_HIP(hipMemcpyAsync(&cnt, pos.p + nk, 4, hipMemcpyDeviceToHost, s));
  TB_HIP(hipMemcpyAsync(&f, flag.p, 4, hipMemcpyDeviceToHost, s));
  ctx->sync();
  *bad = *bad || f != 0;
  return cnt;
}

void build_offdiag(tribit_ctx* ctx, const uint64_t* d_cols, uint64_t ncols, const uint64_t* d_idxs, uint64_t nidxs,
                   uint64_t n, tribit_graph* g) {
  if (n == 0 || n > 0xFFFFFFFEull) fail(TRIBIT_ERR_TOO_LARGE, "vertex count must be in [1, 2^32-2]");
  hipStream_t s = ctx->stream;
  g->ctx = ctx;
  g->n = n;
  g->entries = ncols + nidxs;
  bool bad = false;
  // H: the idxs edges as a CSR by the smaller id
  DevBuf<uint64_t> hk(ctx, nidxs ? nidxs : 1);
  const uint64_t mh = sort_unique(ctx, d_idxs, nidxs, n, hk.p, &bad);
  if (mh > 0xFFFFFFFFull) fail(TRIBIT_ERR_TOO_LARGE, "more than 2^32-1 index edges in one task");
  DevBuf<uint32_t> col(ctx, mh ? mh : 1, kKept), row_ptr(ctx, n + 1, kKept);
  {
    DevBuf<uint32_t> odeg(ctx, n + 1);
    k_fill_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(odeg.p, n + 1, 0u);
    if (mh) k_csr_split<<<grid_for(mh, kBlock), kBlock, 0, s>>>(hk.p, mh, 32, col.p, nullptr, odeg.p);
    scan_u32(ctx, odeg.p, row_ptr.p, n + 1);
  }
  hk.reset();
  // the cols edges, owner first, distinct, as streamed ranges of H rows grouped by owner
  uint64_t mc = 0;
  DevBuf<uint64_t> ck(ctx, ncols ? ncols : 1);
  if (ncols) {
    DevBuf<uint32_t> flag(ctx, 1);
    k_fill_u32<<<1, 64, 0, s>>>(flag.p, 1, 0u);
    k_validate<<<grid_for(ncols, kBlock), kBlock, 0, s>>>(d_cols, ncols, n, flag.p);
    uint32_t f = 0;
    TB_HIP(hipMemcpyAsync(&f, flag.p, 4, hipMemcpyDeviceToHost, s));
    ctx->sync();
    if (f) fail(TRIBIT_ERR_RANGE, "edge key is not (min < max < n)");
    DevBuf<uint64_t> ok(ctx, ncols);
    k_offdiag_keys<<<grid_for(ncols, kBlock), kBlock, 0, s>>>(d_cols, ncols, row_ptr.p, ok.p);
    // owner-first keys are no longer (min < max): dedup without the range check
    DevBuf<uint64_t> sorted(ctx, ncols);
    sort_keys(ctx, ok.p, sorted.p, ncols, 32 + bits_for(n));
    ok.reset();
    DevBuf<uint32_t> head(ctx, ncols + 1), pos(ctx, ncols + 1);
    k_head_flags<<<grid_for(ncols, kBlock), kBlock, 0, s>>>(sorted.p, ncols, head.p);
    k_fill_u32<<<1, 64, 0, s>>>(head.p + ncols, 1, 0u);
    scan_u32(ctx, head.p, pos.p, ncols + 1);
    k_scatter_heads<<<grid_for(ncols, kBlock), kBlock, 0, s>>>(sorted.p, ncols, pos.p, ck.p);
    uint32_t cnt = 0;
    TB_HIP(hipMemcpyAsync(&cnt, pos.p + ncols, 4, hipMemcpyDeviceToHost, s));
    ctx->sync();
    mc = cnt;
  }
  if (bad) fail(TRIBIT_ERR_RANGE, "edge key is not (min < max < n)");
  DevBuf<uint2> rng(ctx, mc ? mc : 1, kKept);
  DevBuf<uint32_t> pid(ctx, mc ? mc : 1, kKept), fw_ptr(ctx, n + 1, kKept), rv_ptr(ctx, n + 1, kKept);
  DevBuf<uint64_t> w_fw(ctx, n, kKept), w_rv(ctx, n, kKept);
  {
    DevBuf<uint32_t> rv_cnt(ctx, n + 1);
    k_fill_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(rv_cnt.p, n + 1, 0u);
    k_fill_u32<<<grid_for(n + 1, kBlock), kBlock, 0, s>>>(fw_ptr.p, n + 1, 0u);
    k_fill_u64<<<grid_for(n, kBlock), kBlock, 0, s>>>(reinterpret_cast<unsigned long long*>(w_fw.p), n);
    k_fill_u64<<<grid_for(n, kBlock), kBlock, 0, s>>>(reinterpret_cast<unsigned long long*>(w_rv.p), n);
    if (mc)
      k_rv_fill<<<grid_for(mc, kBlock), kBlock, 0, s>>>(ck.p, mc, row_ptr.p, rng.p, pid.p, rv_cnt.p,
                                                        reinterpret_cast<unsigned long long*>(w_rv.p));
    scan_u32(ctx, rv_cnt.p, rv_ptr.p, n + 1);
  }
  ck.reset();
  // totals: streamed elements, owner rows
  DevBuf<RowStats> st(ctx, 1);
  k_fill_u32<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t*>(st.p), sizeof(RowStats) / 4, 0u);
  k_sum_u64<<<totals_grid(n), kBlock, 0, s>>>(reinterpret_cast<const unsigned long long*>(w_rv.p), n,
                                              &st.p->wplus);
  k_rows<<<totals_grid(n), kBlock, 0, s>>>(row_ptr.p, nullptr, nullptr, n, st.p, nullptr, false);
  RowStats hst;
  TB_HIP(hipMemcpyAsync(&hst, st.p, sizeof(hst), hipMemcpyDeviceToHost, s));
  ctx->sync();
  g->m = mh;
  g->row_ptr = row_ptr.release();
  g->col = col.release();
  g->relabeled = 0;
  g->m_fwd = 0;
  g->rng_dir = rng.release();
  g->pid_dir = pid.release();
  g->fw_ptr = fw_ptr.release();
  g->rv_ptr = rv_ptr.release();
  g->w_fw = w_fw.release();
  g->w_rv = w_rv.release();
  g->wplus = hst.wplus;  // streamed elements of the task
  g->rows_active = hst.rows_active;
  g->max_outdeg = hst.max_outdeg;
  g->offdiag_lists = mc;
  g->bytes = 4 * (n + 1) * 3 + 4 * (mh ? mh : 1) + 12 * (mc ? mc : 1) + 16 * n;
}

// Releases every device buffer of a graph (the struct stays).
void free_graph_memory(tribit_graph* g) {
  if (!g || !g->ctx) return;
  free_tiles(g);
  core_release(g);
  blocks_release(g);
  bucket_cache_free(g);
  g->ctx->free(g->row_ptr);
  g->ctx->free(g->col);
  g->ctx->free(g->deg);
  g->ctx->free(g->labels);
  g->labels = nullptr;
  g->ctx->free(g->rng_sfx);
  g->ctx->free(g->col16);
  g->col16 = nullptr;
  g->ctx->free(g->sfx_dh);
  g->sfx_dh = nullptr;
  g->ctx->free(g->sfx_split);
  g->sfx_split = nullptr;
  g->ctx->free(g->sfx_ptr);
  g->ctx->free(g->w_sfx);
  g->rng_sfx = nullptr;
  g->sfx_ptr = nullptr;
  g->w_sfx = nullptr;
  g->ctx->free(g->wrow);
  g->ctx->free(g->rng_all);
  g->ctx->free(g->rng_dir);
  g->ctx->free(g->pid_dir);
  g->pid_dir = nullptr;
  g->ctx->free(g->fw_ptr);
  g->ctx->free(g->rv_ptr);
  g->ctx->free(g->w_fw);
  g->ctx->free(g->w_rv);
  g->row_ptr = g->col = g->deg = g->fw_ptr = g->rv_ptr = nullptr;
  g->wrow = g->w_fw = g->w_rv = nullptr;
  g->rng_all = g->rng_dir = nullptr;
}


void free_graph(tribit_graph* g) {
  if (!g) return;
  free_graph_memory(g);
  delete g;
}

}  // namespace tb
