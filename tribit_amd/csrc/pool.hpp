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
// Segments: buffers of one call share segments that are cut up, a quarter of the
// device at most; beyond that, and for the large buffers that an object keeps, a
// buffer gets a segment of its own, which serves later ones of up to an eighth
// less. What a call shared is wholly free when it returns, so no graph or batch
// pins more than the segments it lies in (of at most 128 MiB for its smaller
// buffers).
// Bound: at most three quarters of the device stay free in the pool, more is given
// back by whole segments: what cannot be, because a block in it is in use, lies in
// shared segments and is less than a quarter of the device. A build that needs
// more maps memory anew on each call; R-MAT scale 27 (2.1G edges, 122 GB) builds
// in 0.32 s with its memory kept and took 2.2-2.6 s without.
// No room: the context's own free segments are given back, then those of the
// device's other contexts, then any free block that fits serves; the context's
// shutdown gives back the rest.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <iterator>
#include <map>
#include <mutex>
#include <set>
#include <utility>

namespace tb {

class DevicePool {
 public:
  DevicePool() = default;
  DevicePool(const DevicePool&) = delete;
  DevicePool& operator=(const DevicePool&) = delete;
  ~DevicePool() { leave(); }

  void init(int device, hipStream_t stream, uint64_t total) {
    device_ = device;
    stream_ = stream;
    keep_ = total / 4 * 3;
    cut_most_ = total / 4;
    std::lock_guard<std::mutex> lock(all_mu());
    all().insert(this);
  }

  // nullptr when the device has no room; bytes is a multiple of 256. kept: the
  // buffer outlives the call that takes it.
  void* alloc(uint64_t bytes, bool kept) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (void* p = take_or_grow(bytes, kept)) return p;
      give_back(0);
      if (hipStreamSynchronize(stream_) != hipSuccess) return nullptr;
      if (void* p = take_or_grow(bytes, kept)) return p;
    }
    others_give_back();
    std::lock_guard<std::mutex> lock(mu_);
    if (void* p = take_or_grow(bytes, kept)) return p;
    for (int cls = 0; cls < kClasses; ++cls) {
      const auto it = free_[cls].lower_bound({bytes, 0});
      if (it != free_[cls].end()) return take(it, cls, bytes, cls != kWhole);
    }
    return nullptr;
  }

  // Memory of another context's pool goes back there once this context's stream
  // is done with it, memory of no pool (keys that the caller allocated) to the
  // runtime.
  void free(void* ptr) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(ptr);
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (owns(a)) return put(a);
    }
    std::lock_guard<std::mutex> lock(all_mu());
    for (DevicePool* p : all()) {
      if (p == this) continue;
      std::lock_guard<std::mutex> theirs(p->mu_);
      if (!p->owns(a)) continue;
      (void)hipStreamSynchronize(stream_);
      return p->put(a);
    }
    if (hipFreeAsync(ptr, stream_) != hipSuccess) (void)hipGetLastError();
  }

  // No segment is given back while this lives: around a capture of the stream,
  // which would record the release. Nothing may be taken or freed meanwhile.
  std::unique_lock<std::mutex> hold() { return std::unique_lock<std::mutex>(mu_); }

  // Gives every segment back, used or not (the context ends).
  void release() {
    leave();
    std::lock_guard<std::mutex> lock(mu_);
    for (auto& s : segs_) (void)hipFreeAsync(reinterpret_cast<void*>(s.first), stream_);
    segs_.clear();
    blocks_.clear();
    for (auto& f : free_) f.clear();
    free_bytes_ = cut_bytes_ = 0;
  }

 private:
  struct Block {
    uint64_t size;
    uintptr_t seg;
    int cls;
    bool free;
  };
  using Blocks = std::map<uintptr_t, Block>;
  using Free = std::set<std::pair<uint64_t, uintptr_t>>;  // by size
  // Classes of segments: small, middling and large buffers of a call, small and
  // middling ones of an object, and segments handed out whole. Sizes have
  // segments of their own so that a small buffer does not split the space of a
  // large one.
  static constexpr int kKept = 3, kWhole = 5, kClasses = 6;
  static constexpr uint64_t kSmall = 1ull << 20, kMid = 32ull << 20;
  static constexpr uint64_t kSegment[kWhole] = {16ull << 20, 128ull << 20, 0, 16ull << 20, 128ull << 20};  // least
  static constexpr uint64_t kSplit[kWhole] = {256, 64ull << 10, 1ull << 20, 256, 64ull << 10};  // least tail cut off

  static int class_of(uint64_t bytes, bool kept) {
    const int size = bytes < kSmall ? 0 : bytes < kMid ? 1 : 2;
    return kept ? kKept + size : size;  // kKept + 2 is kWhole
  }

  void* take_or_grow(uint64_t bytes, bool kept) {
    if (void* p = take_free(bytes, kept)) return p;
    return grow(bytes, kept) ? take_free(bytes, kept) : nullptr;
  }

  void* take_free(uint64_t bytes, bool kept) {
    const int cls = class_of(bytes, kept);
    const uint64_t most = bytes + bytes / 8;  // of a block taken whole
    auto it = free_[kWhole].lower_bound({bytes, 0});
    if (it != free_[kWhole].end() && it->first <= most) return take(it, kWhole, bytes, false);
    if (cls == kWhole) {
      for (it = free_[2].lower_bound({bytes, 0}); it != free_[2].end() && it->first <= most; ++it)
        if (whole_segment(*it)) return take(it, 2, bytes, false);
      return nullptr;
    }
    it = free_[cls].lower_bound({bytes, 0});
    return it == free_[cls].end() ? nullptr : take(it, cls, bytes, true);
  }

  bool owns(uintptr_t a) const {  // anywhere in a segment
    auto s = segs_.upper_bound(a);
    return s != segs_.begin() && a < std::prev(s)->first + std::prev(s)->second;
  }

  // The block at `a` is free from now on (no block, or a free one: nothing happens).
  void put(uintptr_t a) {
    auto it = blocks_.find(a);
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

  bool whole_segment(const std::pair<uint64_t, uintptr_t>& f) const {
    const auto s = segs_.find(f.second);
    return s != segs_.end() && s->second == f.first;
  }

  // The free block `it` of class cls for `bytes`; with cut, its tail stays free.
  void* take(Free::iterator it, int cls, uint64_t bytes, bool cut) {
    const uintptr_t p = it->second;
    Block& b = blocks_.at(p);
    free_[cls].erase(it);
    free_bytes_ -= b.size;
    if (cut && b.size - bytes >= kSplit[cls]) {
      const Block tail{b.size - bytes, b.seg, cls, true};
      blocks_.emplace(p + bytes, tail);
      free_[cls].insert({tail.size, p + bytes});
      free_bytes_ += tail.size;
      b.size = bytes;
    }
    b.free = false;
    return reinterpret_cast<void*>(p);
  }

  bool grow(uint64_t bytes, bool kept) {
    const uint64_t page = 2ull << 20;
    const int cls = class_of(bytes, kept);
    if (cls != kWhole) {
      const uint64_t size = ((bytes > kSegment[cls] ? bytes : kSegment[cls]) + page - 1) & ~(page - 1);
      if (cut_bytes_ + size <= cut_most_ && map(size, cls)) {
        cut_bytes_ += size;
        return true;
      }
    }
    return map(bytes < kMid ? bytes : (bytes + page - 1) & ~(page - 1), kWhole);
  }

  bool map(uint64_t size, int cls) {
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

  // Gives wholly free segments back, segments of one buffer and the largest
  // first, until at most `keep` bytes are free.
  void give_back(uint64_t keep) {
    for (const int cls : {kWhole, 2, 4, 1, 3, 0})
      for (auto it = free_[cls].end(); it != free_[cls].begin() && free_bytes_ > keep;) {
        --it;
        if (!whole_segment(*it)) continue;
        const uintptr_t p = it->second;
        free_bytes_ -= it->first;
        if (cls != kWhole) cut_bytes_ -= it->first;
        (void)hipFreeAsync(reinterpret_cast<void*>(p), stream_);
        blocks_.erase(p);
        segs_.erase(p);
        it = free_[cls].erase(it);
      }
  }

  // The pools of a process's contexts, for one that finds no room on its device
  // (never destroyed: a context may end after the process's static objects).
  static std::mutex& all_mu() {
    static std::mutex* const mu = new std::mutex;
    return *mu;
  }
  static std::set<DevicePool*>& all() {
    static auto* const pools = new std::set<DevicePool*>;
    return *pools;
  }
  void leave() {
    std::lock_guard<std::mutex> lock(all_mu());
    all().erase(this);
  }
  void others_give_back() {
    std::lock_guard<std::mutex> lock(all_mu());
    for (DevicePool* p : all()) {
      if (p == this || p->device_ != device_) continue;
      std::lock_guard<std::mutex> theirs(p->mu_);
      p->give_back(0);
      (void)hipStreamSynchronize(p->stream_);
    }
  }

  std::mutex mu_;
  int device_ = 0;
  hipStream_t stream_ = nullptr;
  uint64_t keep_ = 0, free_bytes_ = 0;     // most and present bytes free
  uint64_t cut_most_ = 0, cut_bytes_ = 0;  // of the segments that are cut up
  Blocks blocks_;                          // every block by address
  Free free_[kClasses];                    // free blocks
  std::map<uintptr_t, uint64_t> segs_;     // segment -> size
};

}  // namespace tb
