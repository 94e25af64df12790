"""Host-side checks of the native code's own rules: small C++ programs over its headers, built with g++."""
import os
import subprocess


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "tribit_amd", "csrc")
ROCM = ["-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include"]


def run_cpp(tmp_path, source, includes=()):
    """Builds `source` against the library's headers, runs it and returns its output lines."""
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", *includes, "-I", CSRC, str(src), "-o", str(exe)], check=True,
                   timeout=300)
    return subprocess.run([str(exe)], check=True, timeout=300, capture_output=True, text=True).stdout.split("\n")


ENDS = r"""
#include "ends.hpp"
#include <cstdio>
int main() {
  const uint32_t ends[] = {0u, 1u, (1u << 17) - 1, 1u << 17, (1u << 17) + 1, 1u << 31, 4294901760u, 4292870145u, 0xFFFFFFFEu, 0xFFFFFFFFu};
  for (const uint64_t m : {1ull << 18, 16384001ull, 2147450880ull, 0x7FFFFFFFull}) {
    const uint32_t chunk = tb::end_chunk(m, 256);
    for (const uint32_t e : ends) std::printf("%u %u %u\n", e, chunk, tb::end_chunks(e, chunk));
  }
}
"""


def test_counting_tasks_cover_every_endpoint(tmp_path):
    """Chunks of a group's endpoints up to the most that 2^31 - 1 edges have (the complete graph on 65,536 ids among
    them): as many as whole numbers give, none lost to 32 bits."""
    rows = [list(map(int, line.split())) for line in run_cpp(tmp_path, ENDS, ROCM) if line]
    assert len(rows) == 40
    for ends, chunk, got in rows:
        assert 1 << 17 <= chunk <= 1 << 21
        assert got == -(-ends // chunk), (ends, chunk)


# A device of kTotal bytes whose memory is addresses only.
HIP_STUB = r"""
#pragma once
#include <cstdint>
#include <cstddef>
#include <map>
typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorOutOfMemory = 2;
constexpr uint64_t GiB = 1ull << 30, MiB = 1ull << 20, kTotal = 16 * GiB;
inline std::map<uintptr_t, uint64_t>& mapped() { static std::map<uintptr_t, uint64_t> m; return m; }
inline uint64_t mapped_bytes() { uint64_t s = 0; for (auto& x : mapped()) s += x.second; return s; }
inline hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) {
  static uintptr_t next = 1ull << 40;
  if (mapped_bytes() + n > kTotal) return hipErrorOutOfMemory;
  *p = (void*)next;
  mapped()[next] = n;
  next += (n + 4095) / 4096 * 4096;  // neighbours touch: blocks of two segments must not merge
  return hipSuccess;
}
inline hipError_t hipFreeAsync(void* p, hipStream_t) { return mapped().erase((uintptr_t)p) ? hipSuccess : 1; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
"""

POOL = r"""
#include "pool.hpp"
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(0); } } while (0)
int main() {
  const uint64_t keep = kTotal / 4 * 3;
  {  // pieces of one segment, joined again when freed
    tb::DevicePool p;
    p.init(0, nullptr, kTotal);
    std::vector<void*> v;
    for (int i = 0; i < 1000; ++i) v.push_back(p.alloc(256 * (1 + i % 7), false));
    const uint64_t was = mapped_bytes();
    CHECK(was == 16 * MiB);
    for (size_t i = 0; i < v.size(); i += 2) p.free(v[i]);
    for (size_t i = 1; i < v.size(); i += 2) p.free(v[i]);
    void* whole = p.alloc(MiB - 256, false);
    CHECK(whole == v[0] && mapped_bytes() == was);
    p.free(whole);
    p.free(whole);  // a second free of it changes nothing
    p.release();
    CHECK(mapped().empty());
  }
  {  // a kept buffer leaves the segment of a call's buffer free to be given back
    tb::DevicePool p;
    p.init(0, nullptr, kTotal);
    void* call = p.alloc(3 * GiB, false);
    p.free(call);
    void* kept = p.alloc(64 * MiB, true);
    void* big = p.alloc(15 * GiB, false);
    CHECK(kept && big && mapped_bytes() == 15 * GiB + 64 * MiB);
    p.free(big);
    p.free(kept);
    CHECK(mapped_bytes() <= keep);
    void* again = p.alloc(60 * MiB, true);  // within an eighth: the same segment
    CHECK(again == kept);
    p.release();
  }
  {  // another context's free memory serves an allocation that finds no room
    tb::DevicePool a, b, other_device;
    a.init(0, nullptr, kTotal);
    b.init(0, nullptr, kTotal);
    other_device.init(1, nullptr, kTotal);
    a.free(a.alloc(7 * GiB, false));
    void* held = a.alloc(100 * MiB, false);
    CHECK(mapped_bytes() > 7 * GiB);
    void* p = b.alloc(15 * GiB, false);
    CHECK(p && held);
    CHECK(!b.alloc(2 * GiB, false));
    a.release();
    b.release();
    CHECK(mapped().empty());
  }
  {  // another context's block goes back to it, memory of no pool to the runtime; an inner address to nobody
    tb::DevicePool a, b;
    a.init(0, nullptr, kTotal);
    b.init(0, nullptr, kTotal);
    void* p = a.alloc(64 * MiB, false);
    void* foreign = nullptr;
    CHECK(hipMallocAsync(&foreign, MiB, nullptr) == hipSuccess);
    const uint64_t was = mapped_bytes();
    b.free((char*)p + 4096);
    b.free(p);
    CHECK(mapped_bytes() == was && a.alloc(64 * MiB, false) == p);
    b.free(foreign);
    CHECK(mapped_bytes() == was - MiB);
    a.release();
    b.release();
  }
  {  // the last megabytes: a segment smaller than usual, then a free piece of any class
    tb::DevicePool p;
    p.init(0, nullptr, kTotal);
    void* big = p.alloc(3 * GiB, false);
    void* rest = p.alloc(13 * GiB - 8 * MiB, false);
    void* mid = p.alloc(8 * MiB, false);
    CHECK(big && rest && mid && mapped_bytes() == kTotal);
    p.free(big);
    void* first = p.alloc(2 * GiB, false);
    CHECK(first == big);
    void* piece = p.alloc(4 * MiB, true);
    CHECK(piece && mapped_bytes() == kTotal);
    p.release();
  }
  // random calls: blocks never overlap, and free bytes stay below three quarters of the device
  tb::DevicePool p;
  p.init(0, nullptr, kTotal);
  std::mt19937_64 rng(7);
  std::map<uintptr_t, uint64_t> live;
  uint64_t used = 0, refused = 0;
  for (int i = 0; i < 200000; ++i) {
    if (live.empty() || rng() % 100 < 52) {
      uint64_t n = 256ull << (rng() % 23);
      n += n * (rng() % 256) / 256 & ~255ull;
      const bool kept = rng() % 4 == 0;
      void* q = p.alloc(n, kept);
      if (!q) {
        CHECK(used + n > kTotal / 4);  // a shared quarter may hold pieces too small
        ++refused;
        while (used > kTotal / 8) {  // the program gives up what it holds
          auto it = live.begin();
          std::advance(it, rng() % live.size());
          p.free((void*)it->first);
          used -= it->second;
          live.erase(it);
        }
        continue;
      }
      const uintptr_t a = (uintptr_t)q;
      CHECK(a % 256 == 0);
      auto next = live.lower_bound(a);
      CHECK(next == live.end() || next->first >= a + n);
      CHECK(next == live.begin() || std::prev(next)->first + std::prev(next)->second <= a);
      auto seg = std::prev(mapped().upper_bound(a));
      CHECK(a + n <= seg->first + seg->second);
      live[a] = n;
      used += n;
    } else {
      auto it = live.begin();
      std::advance(it, rng() % live.size());
      p.free((void*)it->first);
      used -= it->second;
      live.erase(it);
      // handed out: up to an eighth, or the least tail, more than asked for
      CHECK(mapped_bytes() <= keep + used + used / 8 + live.size() * MiB);
    }
  }
  for (auto& x : live) p.free((void*)x.first);
  CHECK(mapped_bytes() <= keep);
  void* all = p.alloc(kTotal, false);  // nothing in use: all of the device
  CHECK(all);
  p.free(all);
  CHECK(mapped_bytes() <= keep);
  p.release();
  CHECK(mapped().empty());
  std::printf("ok %d\n", refused > 0);
}
"""


def test_pool_bookkeeping(tmp_path):
    """Split, merge, segments of kept buffers, the bound on free bytes, and what is tried when the device is full, on
    a stand-in for the runtime's allocator."""
    stub = tmp_path / "hip"
    stub.mkdir()
    (stub / "hip_runtime.h").write_text(HIP_STUB)
    assert run_cpp(tmp_path, POOL, ["-I", str(tmp_path)])[0] == "ok 1"
