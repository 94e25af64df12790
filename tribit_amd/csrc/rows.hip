// rows.hip -- the oriented rows of a relabelled graph from its distinct edges
// (gfx950): orientation, and the arcs sorted by (u, v), by partition.
//
// No counterpart in the reference. A radix sort of the arcs (50 bits at 2^25 ids)
// streams them eight times through HBM after a pass that only turns edges into
// arcs, and a pass that splits them follows: 34 ms for the 523M edges of R-MAT
// scale 25, where the kernels here take 25.9; at 2^13 ids and 80K edges 13 launches
// of 60 us against five of 31. Rows have a known upper bound: in degree order no
// outdegree passes deg(u) nor 2 sqrt(m) (the vertices above u have at least its
// degree, octave ids half of it), so the scan P of min(deg(u), 2 sqrt(m)) gives
// every run of rows a place large enough, without counting. Edges become arcs on
// their way into slots of consecutive rows (one or two passes, places by atomics:
// the order inside a slot is free), and each slot is sorted in LDS and written to
// its final place.
//   slots: the positions [0, 2m] of P are cut into quanta of Q; slot 2q holds the
//     rows whose P lies in quantum q, but slot 2q + 1 the last of them if it ends
//     beyond q and its bound is kRowLong or more. An even slot has fewer than
//     Q + kRowLong positions, which is what LDS sorts; an odd one is a single row,
//     sorted through a bitmap of the ids after it if it is longer than that.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include <rocprim/block/block_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include "common.hpp"
#include "device.hpp"
#include "zero.hpp"

namespace tb {

constexpr unsigned kBlock = 256;
constexpr uint32_t kRowThreads = 512;
constexpr uint32_t kRowItems = 12;                        // items per thread of a partition tile: two blocks per CU
// Fewer than kRowFew edges fill the chip only with smaller tiles: k_row_split at
// 80K edges 8.5 us (18 with 12 items); at 2.4M edges both take the same in sum.
constexpr uint32_t kRowItemsFew = 3;
constexpr uint64_t kRowFew = 1ull << 21;
constexpr uint32_t kRowQBits = 12;
// Few edges get smaller slots, whose sorts are shorter and fill more of the chip:
// k_row_sort at 80K edges 9 us with Q = 2^10, 19 with 2^12.
constexpr uint32_t kRowQFew = 10;
constexpr uint32_t kRowLong = 512;
constexpr uint32_t kRowSorted = (1u << kRowQBits) + kRowLong;  // arcs sorted in LDS: 36 KiB, four blocks per CU
constexpr uint32_t kRowSlots = 1032;                      // slots one pass tells apart, with room at the ends
constexpr uint32_t kRowTop = 1024;                        // first step of a search among them
constexpr uint32_t kRowWindow = 1u << 18;                 // ids of a long row's bitmap: 32 KiB
static_assert(2 * kRowsMaxEdges >> kRowQBits <= kRowWindow, "a long row's ids fit the bitmap");

struct RowBound {
  const uint32_t* deg;
  uint64_t n;
  uint32_t most;
  __host__ __device__ uint32_t operator()(uint64_t u) const {
    return u < n ? (deg[u] < most ? deg[u] : most) : 0u;
  }
};

struct Count {
  const uint32_t* c;
  uint64_t n;
  __host__ __device__ uint32_t operator()(uint64_t i) const { return i < n ? c[i] : 0u; }
};

// first[j] of the slots of Q = 2^qb over positions [0, limit]: the first row of
// slot j; first[2 nq] = n.
__global__ void k_row_slots(const uint32_t* __restrict__ P, uint64_t n, uint32_t limit, uint32_t qb,
                            uint32_t* __restrict__ first, ZeroSpans z) {
  const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  z.clear(v);
  if (v > n) return;
  const uint32_t nq = (limit >> qb) + 1;
  const uint32_t p = P[v], pp = v ? P[v - 1] : 0u;
  const uint32_t q = v < n ? p >> qb : nq;
  const uint32_t from = v ? (pp >> qb) + 1 : 0u;  // quanta [from, q] begin at v
  if (from > q) return;
  if (v) first[2 * (from - 1) + 1] = (uint32_t)v - (p - pp >= kRowLong ? 1u : 0u);
  for (uint32_t k = from; k <= q; ++k) {
    first[2 * k] = (uint32_t)v;
    if (k < q) first[2 * k + 1] = (uint32_t)v;
  }
}

// The slot of row u among first[0, nd): the last one that begins at or before u
// (first[0] <= u). Steps of fixed size from `top`, a power of two of at least
// nd / 2, so that the searches of several items run side by side.
__device__ __forceinline__ uint32_t slot_of(const uint32_t* first, uint32_t nd, uint32_t u, uint32_t top) {
  uint32_t at = 0;
  for (uint32_t step = top; step; step >>= 1) {
    const uint32_t i = at + step;
    at = i < nd && first[min(i, nd - 1)] <= u ? i : at;
  }
  return at;
}

template <uint32_t ITEMS>
struct RowLds {
  uint64_t item[ITEMS * kRowThreads];
  uint16_t dig[ITEMS * kRowThreads];
  uint32_t first[kRowSlots], hist[kRowSlots], rel[kRowSlots], end[kRowSlots];
  uint32_t wsum[kRowThreads / 64];
};

// A tile's arcs to the places of their slots: dr = slot << 16 | rank in the tile
// (all ones: none). hist holds the slots' counts; base / end their positions.
template <uint32_t ITEMS>
__device__ __forceinline__ void row_tile(RowLds<ITEMS>& s, const uint64_t (&h)[ITEMS], const uint32_t (&dr)[ITEMS],
                                         uint32_t nd, const uint32_t* __restrict__ base_of,
                                         uint32_t* __restrict__ cursor, uint64_t* __restrict__ out,
                                         uint32_t* __restrict__ flag) {
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < nd; d += kRowThreads) {
    const uint32_t c = s.hist[d];
    if (!c) continue;
    const uint32_t at = base_of[s.first[d]] + atomicAdd(&cursor[d], c);
    if (at + c > s.end[d]) atomicOr(flag, 1u);  // no row passes its bound
    s.rel[d] = at;
  }
  __syncthreads();
  const uint32_t per = (nd + kRowThreads - 1) / kRowThreads, i0 = threadIdx.x * per, lane = lane_id();
  uint32_t sum = 0;
  for (uint32_t i = i0; i < min(i0 + per, nd); ++i) sum += s.hist[i];
  uint32_t inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o);
    if (lane >= (uint32_t)o) inc += t;
  }
  if (lane == 63) s.wsum[threadIdx.x >> 6] = inc;
  __syncthreads();
  uint32_t at = inc - sum, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < kRowThreads / 64; ++w) {
    const uint32_t t = s.wsum[w];
    at += w < (threadIdx.x >> 6) ? t : 0u;
    total += t;
  }
  for (uint32_t i = i0; i < min(i0 + per, nd); ++i) {
    const uint32_t c = s.hist[i];
    s.hist[i] = at;
    s.rel[i] -= at;
    at += c;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j)
    if (dr[j] != 0xFFFFFFFFu) {
      const uint32_t slot = s.hist[dr[j] >> 16] + (dr[j] & 0xFFFFu);
      s.item[slot] = h[j];
      s.dig[slot] = (uint16_t)(dr[j] >> 16);
    }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < total; i += kRowThreads) {
    const uint32_t d = s.dig[i], to = s.rel[d] + i;
    if (to < s.end[d]) out[to] = s.item[i];
  }
}

// First pass: every distinct edge becomes its arc u -> v, u < v the new ids,
// packed (u << kb) | v, in its slot. Bound by the two label gathers per edge (the
// 134 MB of labels at 2^25 ids sit in the last-level cache): 11.0 to 11.4 ms for 523M
// edges, where the gathers alone took 13.1 with one edge per thread.
template <uint32_t ITEMS>
__global__ void __launch_bounds__(kRowThreads) k_row_split(const uint64_t* __restrict__ keys, uint64_t m,
                                                           const uint32_t* __restrict__ lab, uint32_t kb,
                                                           const uint32_t* __restrict__ first, uint32_t nd,
                                                           const uint32_t* __restrict__ P,
                                                           uint32_t* __restrict__ cursor, uint64_t* __restrict__ out,
                                                           uint32_t* __restrict__ flag) {
  __shared__ RowLds<ITEMS> s;
  const uint64_t low = (1ull << kb) - 1, t0 = (uint64_t)blockIdx.x * (ITEMS * kRowThreads) + threadIdx.x;
  uint64_t h[ITEMS];
  uint32_t dr[ITEMS], a[ITEMS], b[ITEMS];
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const uint64_t i = t0 + (uint64_t)j * kRowThreads;
    h[j] = i < m ? keys[i] : kSentinel;
  }
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const bool ok = t0 + (uint64_t)j * kRowThreads < m;
    a[j] = ok ? lab[(uint32_t)(h[j] >> kb)] : 0u;
    b[j] = ok ? lab[(uint32_t)(h[j] & low)] : 0u;
  }
  for (uint32_t i = threadIdx.x; i < nd; i += kRowThreads) {
    s.first[i] = first[i];
    s.end[i] = P[first[i + 1]];
    s.hist[i] = 0u;
    s.rel[i] = 0u;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const uint32_t u = min(a[j], b[j]), v = max(a[j], b[j]);
    h[j] = ((uint64_t)u << kb) | v;
    dr[j] = slot_of(s.first, nd, u, kRowTop);
  }
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j)
    dr[j] = t0 + (uint64_t)j * kRowThreads < m ? (dr[j] << 16) | atomicAdd(&s.hist[dr[j]], 1u) : 0xFFFFFFFFu;
  row_tile(s, h, dr, nd, P, cursor, out, flag);
}

// Second pass, 5.1 ms for 523M arcs (8.4 GB, 1.9 at the rate of a copy; a tile's
// barriers and two blocks per CU are the rest): tile blockIdx.x of first-pass slot blockIdx.y over the fine slots that begin in it.
template <uint32_t ITEMS>
__global__ void __launch_bounds__(kRowThreads) k_row_split2(const uint64_t* __restrict__ in, uint32_t kb,
                                                            const uint32_t* __restrict__ first1,
                                                            const uint32_t* __restrict__ cnt1,
                                                            const uint32_t* __restrict__ first, uint32_t nslots,
                                                            const uint32_t* __restrict__ P,
                                                            uint32_t* __restrict__ cursor, uint64_t* __restrict__ out,
                                                            uint32_t* __restrict__ flag) {
  __shared__ RowLds<ITEMS> s;
  const uint32_t d1 = blockIdx.y, u0 = first1[d1], u1 = first1[d1 + 1], p0 = P[u0];
  const uint32_t cnt = min(cnt1[d1], P[u1] - p0), t0 = blockIdx.x * (ITEMS * kRowThreads);
  if (t0 >= cnt) return;
  uint64_t h[ITEMS];
  uint32_t dr[ITEMS];
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const uint32_t i = t0 + threadIdx.x + j * kRowThreads;
    h[j] = i < cnt ? in[p0 + i] : 0ull;
  }
  uint32_t top = 1;
  while (top < nslots) top <<= 1;
  const uint32_t j0 = slot_of(first, nslots, u0, top), nd = slot_of(first, nslots, u1 - 1, top) - j0 + 1;
  for (uint32_t i = threadIdx.x; i < nd; i += kRowThreads) {
    s.first[i] = first[j0 + i];
    s.end[i] = P[first[j0 + i + 1]];
    s.hist[i] = 0u;
    s.rel[i] = 0u;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) dr[j] = slot_of(s.first, nd, (uint32_t)(h[j] >> kb), kRowTop);
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j)
    dr[j] = t0 + threadIdx.x + j * kRowThreads < cnt ? (dr[j] << 16) | atomicAdd(&s.hist[dr[j]], 1u) : 0xFFFFFFFFu;
  row_tile(s, h, dr, nd, P, cursor + j0, out, flag);
}

// Where the sorted arcs of a slot go.
struct RowOut {
  uint64_t* arcs;    // packed (u << kb) | v
  uint32_t* col;
  uint16_t* col16;   // low 16 bits of v, or null
  uint32_t* odeg;
  uint32_t* flag;    // set when a row breaks the rules its place relies on
};

// A slot's c arcs sorted by (u, v) with IPT items a thread: keys (u - u0, v - u0)
// of only as many bits as the slot's rows and the ids after them need.
template <typename Key, int IPT>
struct RowSort {
  using Sort = rocprim::block_radix_sort<Key, kRowThreads, IPT, rocprim::empty_type, 1, 1, sizeof(Key) == 8 ? 8 : 7,
                                         rocprim::block_radix_rank_algorithm::match>;
  typename Sort::storage_type tmp;
  __device__ __forceinline__ void run(const uint64_t* __restrict__ in, uint32_t c, uint32_t base, uint32_t u0,
                                      uint32_t ubits, uint32_t vbits, uint32_t kb, const RowOut& o) {
    const uint64_t low = (1ull << kb) - 1, vlow = (1ull << vbits) - 1;
    Key k[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) {  // the order inside a slot is free: striped reads
      const uint32_t i = threadIdx.x + j * kRowThreads;
      const uint64_t x = i < c ? in[i] : 0ull;
      k[j] = i < c ? (Key)((((x >> kb) - u0) << vbits) | ((x & low) - u0)) : (Key)~0ull;
    }
    Sort().sort_to_striped(k, tmp, 0, ubits + vbits);
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint32_t i = threadIdx.x + j * kRowThreads;
      const bool ok = i < c;
      const uint32_t u = ok ? (uint32_t)((uint64_t)k[j] >> vbits) + u0 : 0xFFFFFFFFu;
      if (ok) {
        const uint32_t v = (uint32_t)(k[j] & vlow) + u0;
        o.arcs[base + i] = ((uint64_t)u << kb) | v;
        o.col[base + i] = v;
        if (o.col16) o.col16[base + i] = (uint16_t)v;
      }
      const uint32_t run = wave_run_length(u, ok);
      if (run) atomicAdd(&o.odeg[u], run);
    }
  }
};

// The sizes a slot's c arcs are sorted at: at most a third of the keys are padding.
template <typename Key>
union RowSorts {
  RowSort<Key, 1> s1;
  RowSort<Key, 2> s2;
  RowSort<Key, 3> s3;
  RowSort<Key, 4> s4;
  RowSort<Key, 6> s6;
  RowSort<Key, 9> s9;
  template <typename... A>
  __device__ __forceinline__ void run(const uint64_t* __restrict__ in, uint32_t c, A&&... a) {
    if (c <= kRowThreads)
      s1.run(in, c, a...);
    else if (c <= 2 * kRowThreads)
      s2.run(in, c, a...);
    else if (c <= 3 * kRowThreads)
      s3.run(in, c, a...);
    else if (c <= 4 * kRowThreads)
      s4.run(in, c, a...);
    else if (c <= 6 * kRowThreads)
      s6.run(in, c, a...);
    else
      s9.run(in, c, a...);
  }
};
static_assert(kRowSorted == 9 * kRowThreads, "the largest slot");

// Block j sorts slot j and writes its arcs, columns and row lengths: 9.1 ms for 523M
// arcs (11.5 GB; the ranking passes in LDS are the rest). Bound by LDS and barriers,
// so as many waves as fit: 64 registers (80 without the bound: 9.7 ms), keys of 32
// bits where they suffice, six sizes of sort (four up to 8192 arcs: 14.9 ms).
__global__ void __launch_bounds__(kRowThreads, 8) k_row_sort(const uint64_t* __restrict__ in, uint32_t kb, uint64_t n,
                                                          const uint32_t* __restrict__ first,
                                                          const uint32_t* __restrict__ P,
                                                          const uint32_t* __restrict__ cnt,
                                                          const uint32_t* __restrict__ cbase, uint64_t m, RowOut o) {
  __shared__ union {
    RowSorts<uint64_t> k64;
    RowSorts<uint32_t> k32;
    uint32_t bits[kRowWindow / 32];
  } s;
  __shared__ uint32_t s_w[kRowThreads / 64];
  const uint32_t j = blockIdx.x, u0 = first[j], c = min(cnt[j], P[first[j + 1]] - P[u0]), base = cbase[j];
  if (j == 0 && o.col16 && threadIdx.x < 4 && m + threadIdx.x < col16_ids(m))
    o.col16[m + threadIdx.x] = 0;  // the padding to whole dwords plus one
  if (!c) return;
  in += P[u0];
  if (c <= kRowSorted) {
    const uint32_t ur = first[j + 1] - u0, ubits = 32 - (uint32_t)__clz(ur), vbits = 64 - (uint32_t)__clzll(n - u0);
    if (ubits + vbits <= 32)
      s.k32.run(in, c, base, u0, ubits, vbits, kb, o);
    else
      s.k64.run(in, c, base, u0, ubits, vbits, kb, o);
    return;
  }
  // One long row: its ids are distinct, so a bitmap of the ids after u0 lists them
  // in order. All of those have degree 2^kRowQBits or more, so they are fewer than
  // 2 kRowsMaxEdges / 2^kRowQBits; an id order that breaks this sets the flag.
  const uint64_t low = (1ull << kb) - 1, w0 = (uint64_t)u0 + 1;
  const uint32_t lane = lane_id();
  constexpr uint32_t kWords = kRowWindow / 32, kPer = kWords / kRowThreads;
  for (uint32_t i = threadIdx.x; i < kWords; i += kRowThreads) s.bits[i] = 0u;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < c; i += kRowThreads) {
    const uint64_t x = (in[i] & low) - w0;
    if (x < kRowWindow)
      atomicOr(&s.bits[x >> 5], 1u << (x & 31));
    else
      atomicOr(o.flag, 1u);
  }
  __syncthreads();
  uint32_t sum = 0;
  for (uint32_t k = 0; k < kPer; ++k) sum += __popc(s.bits[threadIdx.x * kPer + k]);
  uint32_t inc = sum;
#pragma unroll
  for (int t = 1; t < 64; t <<= 1) {
    const uint32_t x = __shfl_up(inc, t);
    if (lane >= (uint32_t)t) inc += x;
  }
  if (lane == 63) s_w[threadIdx.x >> 6] = inc;
  __syncthreads();
  uint32_t at = base + inc - sum;
  for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) at += s_w[w];
  for (uint32_t k = 0; k < kPer; ++k)
    for (uint32_t word = s.bits[threadIdx.x * kPer + k]; word; word &= word - 1) {
      const uint32_t v = (uint32_t)(w0 + (threadIdx.x * kPer + k) * 32 + (uint32_t)(__ffs((int)word) - 1));
      o.arcs[at] = ((uint64_t)u0 << kb) | v;
      o.col[at] = v;
      if (o.col16) o.col16[at] = (uint16_t)v;
      ++at;
    }
  if (threadIdx.x == 0) o.odeg[u0] = c;
}

template <typename F>
static void scan_to(tribit_ctx* ctx, F f, uint64_t n, uint32_t* out) {
  hipStream_t s = ctx->stream;
  if (n <= kSmallScan) {
    k_scan_block<F><<<1, kScanBlockThreads, 0, s>>>(f, (uint32_t)n, out);
    return;
  }
  const auto it = rocprim::make_transform_iterator(rocprim::counting_iterator<uint64_t>(0), f);
  size_t bytes = 0;
  TB_HIP(rocprim::exclusive_scan(nullptr, bytes, it, out, 0u, (size_t)(n + 1), rocprim::plus<uint32_t>(), s));
  DevBuf<uint8_t> tmp(ctx, bytes ? bytes : 8);
  TB_HIP(rocprim::exclusive_scan(tmp.p, bytes, it, out, 0u, (size_t)(n + 1), rocprim::plus<uint32_t>(), s));
}

void load_rows(tribit_ctx* ctx) { load_code(ctx, kRowsFile, reinterpret_cast<const void*>(k_row_sort)); }

// The arcs of a relabelled graph sorted by (u, v): packed into arcs[m] (whose
// memory may hold the edges: they are read before), col, col16 (or null) and the
// rows' lengths odeg (zeroed before). Every allocation comes before the first write
// to them, so a caller may catch NOMEM and sort instead. edges: distinct, packed (lo << kb) | hi of
// input ids; lab: their new ids; deg: degrees by new id. *flag (zeroed before) is
// set if a row passed its bound, which its degrees rule out.
void build_rows(tribit_ctx* ctx, const uint64_t* edges, uint64_t m, const uint32_t* lab, const uint32_t* deg, uint64_t n,
                uint32_t kb, uint64_t* arcs, uint32_t* col, uint16_t* col16, uint32_t* odeg, uint32_t* flag) {
  hipStream_t s = ctx->stream;
  const uint32_t limit = (uint32_t)(2 * m);
  const uint32_t most = (uint32_t)(2.0 * std::sqrt((double)m)) + 1;
  uint32_t qb = kRowQFew;
  while (qb < kRowQBits && (limit >> qb) >= 512) ++qb;
  uint32_t qb1 = qb;
  while ((limit >> qb1) >= 512) ++qb1;
  const bool two = qb1 > qb;
  const uint32_t nq = (limit >> qb) + 1, nslots = 2 * nq, nq1 = (limit >> qb1) + 1, nd1 = 2 * nq1;
  DevBuf<uint32_t> P(ctx, n + 1), first(ctx, (uint64_t)nslots + 1), cnt(ctx, nslots), cbase(ctx, (uint64_t)nslots + 1);
  DevBuf<uint32_t> first1, cnt1;
  scan_to(ctx, RowBound{deg, n, most}, n, P.p);
  if (two) {
    first1 = DevBuf<uint32_t>(ctx, nd1 + 1);
    cnt1 = DevBuf<uint32_t>(ctx, nd1);
    ZeroSpans z{{cnt1.p, nullptr, nullptr}, {nd1, 0, 0}};
    const unsigned grid = grid_for(z.grid_items(n + 1), kBlock);
    k_row_slots<<<grid, kBlock, 0, s>>>(P.p, n, limit, qb1, first1.p, z);
  }
  ZeroSpans z{{cnt.p, nullptr, nullptr}, {nslots, 0, 0}};
  const unsigned grid = grid_for(z.grid_items(n + 1), kBlock);
  k_row_slots<<<grid, kBlock, 0, s>>>(P.p, n, limit, qb, first.p, z);
  DevBuf<uint64_t> b1(ctx, limit), b2;
  if (two) b2 = DevBuf<uint64_t>(ctx, limit);
  const auto split = [&](auto items) {
    constexpr uint32_t kItems = decltype(items)::value, kTile = kItems * kRowThreads;
    k_row_split<kItems><<<grid_for(m, kTile), kRowThreads, 0, s>>>(edges, m, lab, kb, two ? first1.p : first.p,
                                                                   two ? nd1 : nslots, P.p, two ? cnt1.p : cnt.p, b1.p,
                                                                   flag);
    if (!two) return;
    // an even slot has fewer than Q1 + kRowLong positions, an odd one at most `most`
    const uint32_t tiles = (uint32_t)((std::max<uint64_t>((1ull << qb1) + kRowLong, most) + kTile - 1) / kTile);
    k_row_split2<kItems><<<dim3(tiles, nd1), kRowThreads, 0, s>>>(b1.p, kb, first1.p, cnt1.p, first.p, nslots, P.p,
                                                                  cnt.p, b2.p, flag);
  };
  if (m < kRowFew)
    split(std::integral_constant<uint32_t, kRowItemsFew>{});
  else
    split(std::integral_constant<uint32_t, kRowItems>{});
  scan_to(ctx, Count{cnt.p, nslots}, nslots, cbase.p);
  k_row_sort<<<nslots, kRowThreads, 0, s>>>(two ? b2.p : b1.p, kb, n, first.p, P.p, cnt.p, cbase.p, m,
                                            RowOut{arcs, col, col16, odeg, flag});
  TB_HIP(hipGetLastError());
}

}  // namespace tb
