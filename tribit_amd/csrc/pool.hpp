// pool.hpp -- device memory of one context, kept between calls.
//
// Preprocessing takes and gives back about forty buffers per graph. Through the
// runtime's stream-ordered pool each of them cost 0.35-0.4 ms once that pool had
// returned its memory (the release threshold did not hold it), and giving back
// 0.1-4.6 ms: 7.5 ms a call for a 1.1M-edge graph whose kernels run 1.7 ms, and
// 0.5-2.4 s for R-MAT scale 25. Here freed blocks stay with the context, are
// merged with their free neighbours and handed out again.
//
// Order: every use of a block is on its context's one stream, so a block freed
// by the host while a kernel still runs is only written again behind that kernel.
// Bound: free bytes beyond `keep` are given back, whole segments at a time; an
// allocation that fails gives all free segments back and tries again; the
// context's shutdown gives back the rest.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <mutex>
#include <set>
#include <utility>

namespace tb {

class DevicePool {
 public:
  void init(hipStream_t stream, uint64_t keep) {
    stream_ = stream;
    keep_ = keep;
  }

  // nullptr when the device has no room; bytes is a multiple of 256.
  void* alloc(uint64_t bytes) {
    std::lock_guard<std::mutex> lock(mu_);
    const int cls = bytes < kSmall ? 0 : bytes < kMid ? 1 : 2;
    auto it = free_[cls].lower_bound({bytes, 0});
    if (it == free_[cls].end()) {
      if (!grow(cls, bytes)) {
        give_back(0);
        if (hipStreamSynchronize(stream_) != hipSuccess || !grow(cls, bytes)) return nullptr;
      }
      it = free_[cls].lower_bound({bytes, 0});
    }
    const uintptr_t p = it->second;
    Block& b = blocks_.at(p);
    if (b.size - bytes >= kSplit[cls]) {  // the tail stays free
      const Block tail{b.size - bytes, b.seg, cls, true};
      blocks_.emplace(p + bytes, tail);
      free_[cls].insert({tail.size, p + bytes});
      free_bytes_ += tail.size;
    }
    free_[cls].erase(it);
    free_bytes_ -= b.size;
    auto next = std::next(blocks_.find(p));
    if (next != blocks_.end() && next->first == p + bytes) b.size = bytes;
    b.free = false;
    return reinterpret_cast<void*>(p);
  }

  void free(void* ptr) {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = blocks_.find(reinterpret_cast<uintptr_t>(ptr));
    if (it == blocks_.end() || it->second.free) return;
    it->second.free = true;
    free_bytes_ += it->second.size;
    auto next = std::next(it);
    if (next != blocks_.end() && next->second.free && next->second.seg == it->second.seg) merge(it, next);
    if (it != blocks_.begin()) {
      auto prev = std::prev(it);
      if (prev->second.free && prev->second.seg == it->second.seg) {
        merge(prev, it);
        it = prev;
      }
    }
    free_[it->second.cls].insert({it->second.size, it->first});
    if (free_bytes_ > keep_) give_back(keep_);
  }

  // Gives every segment back, used or not (the context ends).
  void release() {
    std::lock_guard<std::mutex> lock(mu_);
    for (auto& s : segs_) (void)hipFreeAsync(reinterpret_cast<void*>(s.first), stream_);
    segs_.clear();
    blocks_.clear();
    for (auto& f : free_) f.clear();
    free_bytes_ = 0;
  }

 private:
  struct Block {
    uint64_t size;
    uintptr_t seg;
    int cls;
    bool free;
  };
  using Blocks = std::map<uintptr_t, Block>;
  // Small, middling and large buffers come from segments of their own, so that
  // a small one that lives long does not split the space of a large one.
  static constexpr uint64_t kSmall = 1ull << 20, kMid = 32ull << 20;
  static constexpr uint64_t kSegment[3] = {16ull << 20, 128ull << 20, 0};  // least segment size
  static constexpr uint64_t kSplit[3] = {256, 64ull << 10, 1ull << 20};    // least tail split off

  bool grow(int cls, uint64_t bytes) {
    uint64_t size = bytes > kSegment[cls] ? bytes : kSegment[cls];
    size = (size + (2ull << 20) - 1) & ~((2ull << 20) - 1);
    void* p = nullptr;
    if (hipMallocAsync(&p, size, stream_) != hipSuccess || !p) {
      (void)hipGetLastError();
      return false;
    }
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    segs_.emplace(a, size);
    blocks_.emplace(a, Block{size, a, cls, true});
    free_[cls].insert({size, a});
    free_bytes_ += size;
    return true;
  }

  // `b` joins the free block `a` before it; neither is left in the free index.
  void merge(Blocks::iterator a, Blocks::iterator b) {
    free_[a->second.cls].erase({a->second.size, a->first});
    free_[b->second.cls].erase({b->second.size, b->first});
    a->second.size += b->second.size;
    blocks_.erase(b);
  }

  // Gives wholly free segments back, the largest first, until at most `keep`
  // bytes are free.
  void give_back(uint64_t keep) {
    for (int cls = 2; cls >= 0; --cls)
      for (auto it = free_[cls].end(); it != free_[cls].begin() && free_bytes_ > keep;) {
        --it;
        const uintptr_t p = it->second;
        auto s = segs_.find(p);
        if (s == segs_.end() || s->second != it->first) continue;
        free_bytes_ -= it->first;
        (void)hipFreeAsync(reinterpret_cast<void*>(p), stream_);
        blocks_.erase(p);
        segs_.erase(s);
        it = free_[cls].erase(it);
      }
  }

  std::mutex mu_;
  hipStream_t stream_ = nullptr;
  uint64_t keep_ = 0, free_bytes_ = 0;
  Blocks blocks_;                                       // every block by address
  std::set<std::pair<uint64_t, uintptr_t>> free_[3];    // free blocks by size, per class
  std::map<uintptr_t, uint64_t> segs_;                  // segment -> size
};

}  // namespace tb
